// Batched executor: many small circuits, each run from |0...0> and reduced to
// the expectation value of its observable, together.
//
// What it replaces: for each circuit, QuantumCircuit::update_quantum_state
// (src/cppsim/circuit.cpp:46-57, one kernel launch and synchronisation per gate
// on the GPU backend) and Observable::get_expectation_value
// (src/cppsim/observable.cpp:56-58 -> general_quantum_operator.cpp:105-141, one
// reduction per term).
//
// Design:
//   * the state lives in LDS, 2^lq complex128 with lq = min(n, 12) (64 KiB at 12 qubits): two
//     work-groups share a CU, and since they drift apart, one's memory phases and sub-operation
//     handling overlap the other's FP64 arithmetic;
//   * a circuit of at most 12 qubits is one work-group, from |0> to its energy; circuits of 13..20
//     qubits keep the state in device memory and are processed in 2^12-amplitude tiles, one
//     "stage" at a time: a stage is a set of gates whose dense part lies in one 12-qubit window
//     (qubits 0..2 are always in the window, so a tile is made of 128-byte contiguous runs;
//     diagonal gates may touch qubits outside, which are constants of a tile);
//   * one launch per stage number covers that stage's tiles of every circuit, in descending cost;
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
// Scheduling (host): see Picker in qm_tile.hpp.
//
// Bound: FP64 issue and the latency of the steps around it (sub-operation decoding, LDS round trips,
// barriers), not HBM: a stage of a 26-qubit brickwork circuit takes 1.13 ms of which its 2.1 GB
// need 0.4 ms.  26 qubits, 10 layers: 9.87 ms with 13 stages of 13-qubit windows picked in
// gate order and one work-group per CU; 6.55 ms with Picker's 5 stages and two work-groups per
// CU; 5.64 ms with shears for three quarters of the matrices (all but the last on a qubit since, see
// reduce_matrices: another 6 % at 20 layers).  QAOA (4 layers, ring and
// chords, 26 qubits): 13.7 -> 10.2 -> 6.0 ms, the last from Z rotations in place of
// diagonals read per amplitude.  512 circuits of 8 to 16 qubits: 1.75 -> 0.69 ms, from one
// work-group per tile instead of per circuit; 0.60 -> 0.43 from energy_sum.
#include <cstring>

#include "qm_tile.hpp"

namespace qm {
namespace {

struct DCirc {
    u32 n, lq, nstage, stage0, term0, nterm;
    u64 state_off;  // complex128 offset of the circuit's state in the scratch buffer
    u32 chunk0;     // first entry of the circuit's partial energies (circuits of several tiles)
    u32 pad;
};
struct DItem {
    u32 circ, tile;
};
// Circuits above this size run in tiles; a tile is 64 KiB, so two work-groups share a CU.
constexpr u32 kTileLocal = QM_BATCH_TILE_QUBITS;
// This thread's share of sum_k c_k Re <psi|P_k|psi> over the `len` amplitudes from x0 on (a power
// of two, aligned), which lie in LDS (swizzled slots); partners beyond them are read from the state in
// device memory.  Threads [0, stride) take part.  Eight amplitudes at a time, the terms in the inner loop:
// a term's eight partners are loaded together, where one amplitude at a time waited for each.  The
// energies of 512 circuits of 8 to 16 qubits (transverse-field Ising chains): those of more than 12
// qubits 224 us with a partner at a time from device memory, 116 with eight (11 TB/s from L2),
// 88 with the tile in LDS, and diagonal terms as one sum of signed coefficients per amplitude.
__device__ __forceinline__ double energy_sum(const double2* __restrict__ gs, const double2* st, const DCirc& c,
                                             const DTerm* __restrict__ terms, u32 x0, u32 len, u32 stride) {
    constexpr int P = 8;
    double acc = 0.0;
    if (threadIdx.x >= stride) return acc;
    auto signed_by = [](double v, u32 bits) {  // (-1)^popcount(bits) v
        return __hiloint2double(__double2hiint(v) ^ (int)(__popc(bits) << 31), __double2loint(v));
    };
    for (u32 first = threadIdx.x; first < len; first += P * stride) {
        u32 x[P], slot[P];
        double2 px[P];
        double diag[P];  // sum of the diagonal terms' signed coefficients
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const u32 at = first + (u32)i * stride;
            x[i] = at < len ? at : 0;  // an amplitude of 0 behind the end
            slot[i] = slot_of(x[i]);
            px[i] = st[slot[i]];
            if (at >= len) px[i] = make_double2(0.0, 0.0);
            x[i] += x0;
            diag[i] = 0.0;
        }
        for (u32 k = 0; k < c.nterm; ++k) {
            const DTerm tm = terms[c.term0 + k];
            const u32 bf = (u32)tm.bf, pf = (u32)tm.pf;
            // Re(z i^rot): z.x, -z.y, -z.x, z.y with z = psi_x conj(psi_y)
            const double coef = ((tm.rot + 1u) & 2u) ? -tm.coef : tm.coef;
            if (bf == 0) {
                if (tm.rot & 1u) continue;  // the imaginary part of |psi_x|^2
#pragma unroll
                for (int i = 0; i < P; ++i) diag[i] += signed_by(coef, x[i] & pf);
                continue;
            }
            double2 py[P];
            if (bf < len) {
                const u32 sb = slot_of(bf);
#pragma unroll
                for (int i = 0; i < P; ++i) py[i] = st[slot[i] ^ sb];
            } else {
#pragma unroll
                for (int i = 0; i < P; ++i) py[i] = gs[x[i] ^ bf];
            }
            if (tm.rot & 1u) {
#pragma unroll
                for (int i = 0; i < P; ++i) py[i] = make_double2(-py[i].y, py[i].x);
            }
            if (pf) {
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    py[i].x = signed_by(py[i].x, x[i] & pf);
                    py[i].y = signed_by(py[i].y, x[i] & pf);
                }
            }
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i < P; ++i) sum = fma(px[i].x, py[i].x, fma(px[i].y, py[i].y, sum));
            acc = fma(coef, sum, acc);
        }
#pragma unroll
        for (int i = 0; i < P; ++i) acc = fma(diag[i], fma(px[i].x, px[i].x, px[i].y * px[i].y), acc);
    }
    return acc;
}

template <int K>
constexpr u32 tile_threads() { return K == 4 ? 256u : 512u; }

// Stage `level` of every circuit that has one, a work-group per (circuit, tile): a circuit of at
// most 12 qubits is one tile and one stage, from |0> to its energy in LDS; a larger one keeps its
// state in device memory.  The tiles of a stage are independent, so a 16-qubit circuit is 16
// work-groups of a launch instead of one work-group's loop over them: 512 circuits of 8 to 16
// qubits, 4 to 8 layers, were bound by that chain on the largest ones.
template <int K>
__global__ __launch_bounds__(tile_threads<K>(), K == 4 ? 2 : 4) void k_batch_level(
    const DCirc* __restrict__ circs, const DStage* __restrict__ stages, const DPass* __restrict__ passes,
    const DSub* __restrict__ subs, const double2* __restrict__ pool, const DTerm* __restrict__ terms,
    const DItem* __restrict__ items, u32 level, double2* __restrict__ scratch, double* __restrict__ energies, int keep) {
    extern __shared__ double2 st[];
    __shared__ u32 hi_tab[1u << (kTileLocal - kLowFixed)];
    __shared__ double red[16];
    const u32 tid = threadIdx.x, bd = blockDim.x;
    const DItem it = items[blockIdx.x];
    const DCirc c = circs[it.circ];
    const DStage sg = stages[c.stage0 + level];
    const u32 lq = c.lq, L = 1u << lq, tl = c.n - lq;
    double2* gs = scratch + c.state_off;
    const u64 tb = tile_base(it.tile, tl, sg);
    if (tl > 0) {
        build_hi_tab(hi_tab, lq, sg);
        __syncthreads();
    }
    if (sg.npass) warm_program(passes[sg.pass0], subs, pool);  // a circuit without gates has no pass to read
    if (level == 0) {
        // |0...0>: slot_of(0) == 0 and amplitude 0 lies in tile 0
        for (u32 i = tid; i < L; i += bd) st[i] = make_double2((i == 0 && it.tile == 0) ? 1.0 : 0.0, 0.0);
    } else {
        for (u32 i = tid; i < L; i += bd) st[slot_of(i)] = gs[tile_index(tb, hi_tab, i)];
    }
    __syncthreads();
    run_passes<K, tile_threads<K>(), 1>(st, lq, passes, sg.pass0, sg.npass, subs, pool, it.tile);
    if (tl > 0) {
        for (u32 i = tid; i < L; i += bd) gs[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
        return;
    }
    if (keep)
        for (u32 i = tid; i < L; i += bd) gs[i] = st[slot_of(i)];
    // a thread count that depends on the circuit alone: its energy does not depend on the batch
    const u32 part = min(tile_threads<K>(), max(64u, L >> K));
    const double total = block_sum(energy_sum(gs, st, c, terms, 0, L, part), red);
    if (tid == 0) energies[it.circ] = total;
}

// Energies of the circuits of several tiles: partial sums over 2^12 amplitudes, then one thread per
// circuit adds them in order.
constexpr u32 kEnergyThreads = 512;
__global__ __launch_bounds__(kEnergyThreads) void k_batch_energy(const DCirc* __restrict__ circs, const DTerm* __restrict__ terms,
                                                      const DItem* __restrict__ items, const double2* __restrict__ scratch,
                                                      double* __restrict__ partials) {
    extern __shared__ double2 st[];
    __shared__ double red[16];
    const DItem it = items[blockIdx.x];
    const DCirc c = circs[it.circ];
    const u32 x0 = it.tile << kTileLocal, len = 1u << min(c.n, kTileLocal);
    const double2* gs = scratch + c.state_off;
    for (u32 i = threadIdx.x; i < len; i += kEnergyThreads) st[slot_of(i)] = gs[x0 + i];
    __syncthreads();
    const double total = block_sum(energy_sum(gs, st, c, terms, x0, len, kEnergyThreads), red);
    if (threadIdx.x == 0) partials[c.chunk0 + it.tile] = total;
}
__global__ __launch_bounds__(64) void k_batch_finish(const DCirc* __restrict__ circs, const u32* __restrict__ large,
                                                     u32 nlarge, const double* __restrict__ partials,
                                                     double* __restrict__ energies) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlarge) return;
    const DCirc c = circs[large[i]];
    const u32 chunks = c.n > kTileLocal ? 1u << (c.n - kTileLocal) : 1u;
    double e = 0.0;
    for (u32 k = 0; k < chunks; ++k) e += partials[c.chunk0 + k];
    energies[large[i]] = e;
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
        run_passes<K, T, stage_blocks<K>()>(st, lq, passes, sg.pass0, sg.npass, subs, pool, t);
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
    // (Windows below 13 qubits come here at K = 2 only; the others run in k_tile.  Their branches stay
    // at K = 3 and 4 all the same: compiled without them the 13-qubit path is 4 to 19 % slower, e.g.
    // K = 4, a Fourier transform on 26 qubits 7.8 -> 9.1 ms.)
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
        run_passes<K, T, stage_blocks<K>()>(st, lq, passes, sg.pass0, sg.npass, subs, pool, t);
        for (u32 i = threadIdx.x; i < L; i += T) state[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
        __syncthreads();
    }
}

// A grid has fewer than 2^32 threads, and 34 qubits in windows of 8 are 2^26 tiles of 64: the
// tiles of a stage go out in launches of this many.
constexpr u64 kTilesPerLaunch = 1ULL << 20;

// One stage of a single-state circuit with a work-group per tile (tiles from tile0 on) of at most 2^12 amplitudes: two or more groups share a
// CU and drift apart, so one's memory phase overlaps another's passes without a prefetch.
template <int K>
__global__ __launch_bounds__(tile_threads<K>(), K == 4 ? 2 : 4) void k_tile(double2* __restrict__ state, u32 lq, u32 tl,
                                                                            u64 tile0, DStage sg,
                                                                            const DPass* __restrict__ passes,
                                                                            const DSub* __restrict__ subs,
                                                                            const double2* __restrict__ pool) {
    extern __shared__ double2 st[];
    __shared__ u64 hi_tab[1u << (kTileLocal - kLowFixed)];
    constexpr u32 T = tile_threads<K>();
    const u32 L = 1u << lq;
    build_hi_tab(hi_tab, lq, sg);
    const u64 tile = tile0 + blockIdx.x;
    const u64 tb = tile_base(tile, tl, sg);
    __syncthreads();
    constexpr u32 P = (1u << kTileLocal) / T;
    if (L == P * T) {
        double2 r[P];
#pragma unroll
        for (u32 k = 0; k < P; ++k) r[k] = state[tile_index(tb, hi_tab, threadIdx.x + k * T)];
        warm_program(passes[sg.pass0], subs, pool);  // while the tile is on its way
#pragma unroll
        for (u32 k = 0; k < P; ++k) st[slot_of(threadIdx.x + k * T)] = r[k];
    } else {
        warm_program(passes[sg.pass0], subs, pool);
        for (u32 i = threadIdx.x; i < L; i += blockDim.x) st[slot_of(i)] = state[tile_index(tb, hi_tab, i)];
    }
    __syncthreads();
    run_passes<K, T, 1>(st, lq, passes, sg.pass0, sg.npass, subs, pool, tile);
    if (L == P * T) {
#pragma unroll
        for (u32 k = 0; k < P; ++k) {
            const u32 i = threadIdx.x + k * T;
            state[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
        }
    } else {
        for (u32 i = threadIdx.x; i < L; i += blockDim.x) state[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
    }
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

}  // namespace
// A circuit ready to join a batch (batch_add_prepared).
struct PreparedCircuit {
    HCirc c;
};
}  // namespace qm

struct qm_batch {
    std::vector<qm::HCirc> circs;
    // compiled
    int device = -1;
    char* d_program = nullptr;  // one allocation, filled by one copy: the arrays of the next seven and d_large
    unsigned K = 0;
    int keep = 0;
    std::vector<qm::DCirc> h_circs;
    qm::u64 n_stages = 0, n_passes = 0, n_subs = 0;
    qm::DCirc* d_circs = nullptr;
    qm::DStage* d_stages = nullptr;
    qm::DPass* d_passes = nullptr;
    qm::DSub* d_subs = nullptr;
    double2* d_pool = nullptr;
    qm::DTerm* d_terms = nullptr;
    qm::DItem* d_items = nullptr;     // the launches' items one after another, then the energy items
    qm::u32* d_large = nullptr;       // circuits of several tiles
    double2* d_scratch = nullptr;
    double* d_energies = nullptr;
    double* d_partials = nullptr;
    struct Level {
        qm::u32 first, count, lq;  // items; the largest tile among them
    };
    std::vector<Level> levels;
    Level energy_items{0, 0, 0};
    qm::u32 n_large = 0;
    size_t cap[4] = {0, 0, 0, 0};  // bytes held: program, scratch, energies, partials
    bool lds_set = false;               // the kernel's LDS limit has been raised on this device
    unsigned lq_cap = 13;               // qubits held in LDS per tile, at most kTileLocal (qm_batch_set_local_qubits)
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
        lds_set = false;
        if (device >= 0) {
            (void)hipSetDevice(device);
            void* ptrs[] = {d_program, d_scratch, d_energies, d_partials};
            for (void* p : ptrs)
                if (p) (void)hipFree(p);
        }
        d_program = nullptr; d_circs = nullptr; d_stages = nullptr; d_passes = nullptr; d_subs = nullptr; d_pool = nullptr;
        d_terms = nullptr; d_items = nullptr; d_large = nullptr; d_scratch = nullptr; d_energies = nullptr;
        d_partials = nullptr;
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
    char* d_program = nullptr;  // one allocation, filled by one copy: passes, sub-operations, pool
    qm::DPass* d_passes = nullptr;
    qm::DSub* d_subs = nullptr;
    double2* d_pool = nullptr;
    void release() {
        if (device >= 0) {
            (void)hipSetDevice(device);
            if (d_program) (void)hipFree(d_program);
        }
        d_program = nullptr; d_passes = nullptr; d_subs = nullptr; d_pool = nullptr;
        device = -1;
        per_cu = 0;
    }
};

namespace qm {
namespace {

// Raises the kernel's LDS limit.  Kept out of the launch path so a graph capture only sees
// stream operations.
bool batch_prepare_launch(qm_batch* b, const char* what) {
    const void* fn = b->K == 2   ? (const void*)k_batch_level<2>
                     : b->K == 3 ? (const void*)k_batch_level<3>
                                 : (const void*)k_batch_level<4>;
    if (!hip_ok(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(double2) << kTileLocal)),
                what) ||
        !hip_ok(hipFuncSetAttribute((const void*)k_batch_energy, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)(sizeof(double2) << kTileLocal)),
                what))
        return false;
    b->lds_set = true;
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
    if (!batch_ok(b, "qm_batch_add_circuit")) return -1;
    PreparedCircuit* c = batch_prepare_circuit(n, gates, gate_count, bf, pf, rot, coefs, term_count);
    return c ? batch_add_prepared(b, c) : -1;
}

}  // extern "C"

namespace qm {
PreparedCircuit* batch_prepare_circuit(UINT n, const qm_batch_gate* gates, UINT gate_count, const ITYPE* bf,
                                       const ITYPE* pf, const UINT* rot, const double* coefs, UINT term_count) {
    const char* what = "qm_batch_add_circuit";
    if (n < 1 || n > QM_BATCH_MAX_QUBITS) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: qubit count %u outside 1..%u", what, n, QM_BATCH_MAX_QUBITS);
        return nullptr;
    }
    if ((gate_count && !gates) || (term_count && (!bf || !pf || !rot || !coefs))) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null gate or term array", what);
        return nullptr;
    }
    HCirc c;
    if (!convert_gates(n, gates, gate_count, c, what)) return nullptr;
    for (UINT t = 0; t < term_count; ++t) {
        if ((bf[t] >> n) || (pf[t] >> n)) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: term %u acts beyond %u qubits", what, t, n);
            return nullptr;
        }
        DTerm tm{};
        tm.bf = bf[t];
        tm.pf = pf[t];
        tm.rot = rot[t];
        tm.coef = coefs[t];
        c.terms.push_back(tm);
    }
    return new PreparedCircuit{std::move(c)};
}
int batch_add_prepared(qm_batch* b, PreparedCircuit* c) {
    b->circs.push_back(std::move(c->c));
    delete c;
    return (int)b->circs.size() - 1;
}
u32 batch_prepared_width(const PreparedCircuit* c) {
    size_t most = 0;
    for (const HOp& o : c->c.ops)
        if (o.type == 0) most = std::max(most, o.q.size());
    return (u32)most;
}
void batch_destroy_prepared(PreparedCircuit* c) { delete c; }
}  // namespace qm

extern "C" {

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
    b->drop_graph();  // device buffers and the launches may change
    b->lds_set = false;
    b->h_circs.clear();
    if (!use_device(dev)) return QM_ERR_HIP;
    Flat f;
    std::vector<DTerm> terms;
    std::vector<DCirc> dc;
    u64 state_off = 0;
    const u32 lq_cap = std::min((u32)b->lq_cap, kTileLocal);
    u32 nlevel = 0, nchunk = 0;
    std::vector<u32> large;
    std::vector<DItem> energy;
    for (const HCirc& c : b->circs) {
        DCirc d{};
        d.n = c.ne;
        d.lq = std::min(c.ne, lq_cap);
        d.stage0 = (u32)f.stages.size();
        d.nstage = schedule_circuit(f, c, K, lq_cap);
        d.term0 = (u32)terms.size();
        d.nterm = (u32)c.terms.size();
        terms.insert(terms.end(), c.terms.begin(), c.terms.end());
        d.state_off = state_off;
        if (c.ne > lq_cap || keep_states) state_off += 1ULL << c.ne;
        nlevel = std::max(nlevel, d.nstage);
        if (c.ne > lq_cap) {
            const u32 chunks = c.ne > kTileLocal ? 1u << (c.ne - kTileLocal) : 1u;
            d.chunk0 = nchunk;
            for (u32 k = 0; k < chunks; ++k) energy.push_back({(u32)dc.size(), k});
            nchunk += chunks;
            large.push_back((u32)dc.size());
        }
        dc.push_back(d);
    }
    // each level's items in descending cost (amplitudes x (passes + terms of a single tile), so that
    // the last work-groups of a launch are short ones
    std::vector<DItem> items;
    std::vector<qm_batch::Level> levels;
    for (u32 lv = 0; lv < nlevel; ++lv) {
        std::vector<std::pair<double, u32>> order;
        for (u32 i = 0; i < dc.size(); ++i) {
            if (dc[i].nstage <= lv) continue;
            const double work = f.stages[dc[i].stage0 + lv].npass + (dc[i].n == dc[i].lq ? dc[i].nterm + 1 : 1);
            order.emplace_back(std::ldexp(work, (int)dc[i].lq), i);
        }
        std::stable_sort(order.begin(), order.end(), [](const auto& x, const auto& y) { return x.first > y.first; });
        qm_batch::Level L{(u32)items.size(), 0, kMinQubits};
        for (const auto& o : order) {
            L.lq = std::max(L.lq, dc[o.second].lq);
            for (u32 t = 0; t < 1u << (dc[o.second].n - dc[o.second].lq); ++t) items.push_back({o.second, t});
        }
        L.count = (u32)items.size() - L.first;
        levels.push_back(L);
    }
    const qm_batch::Level energy_items{(u32)items.size(), (u32)energy.size(), 0};
    items.insert(items.end(), energy.begin(), energy.end());
    if (f.pool.empty()) f.pool.push_back(make_double2(0, 0));
    if (f.subs.empty()) f.subs.push_back(DSub{});
    if (f.passes.empty()) f.passes.push_back(DPass{});
    if (terms.empty()) terms.push_back(DTerm{});
    if (items.empty()) items.push_back(DItem{});
    b->device = (int)dev;
    // one copy: a copy command costs some 30 us, which eight arrays paid each
    std::vector<char> host;
    auto put = [&](const auto& v) {
        const size_t at = (host.size() + 255) & ~size_t(255), bytes = v.size() * sizeof(v[0]);
        host.resize(at + bytes);
        if (bytes) std::memcpy(host.data() + at, v.data(), bytes);
        return at;
    };
    const size_t at_circs = put(dc), at_stages = put(f.stages), at_passes = put(f.passes), at_subs = put(f.subs),
                 at_pool = put(f.pool), at_terms = put(terms), at_items = put(items), at_large = put(large);
    bool ok = dev_reserve((void**)&b->d_program, &b->cap[0], host.size(), what) &&
              hip_ok(hipMemcpy(b->d_program, host.data(), host.size(), hipMemcpyHostToDevice), what);
    if (ok) {
        b->d_circs = (DCirc*)(b->d_program + at_circs);
        b->d_stages = (DStage*)(b->d_program + at_stages);
        b->d_passes = (DPass*)(b->d_program + at_passes);
        b->d_subs = (DSub*)(b->d_program + at_subs);
        b->d_pool = (double2*)(b->d_program + at_pool);
        b->d_terms = (DTerm*)(b->d_program + at_terms);
        b->d_items = (DItem*)(b->d_program + at_items);
        b->d_large = (u32*)(b->d_program + at_large);
    }
    if (ok && state_off) {
        ok = dev_reserve((void**)&b->d_scratch, &b->cap[1], state_off * sizeof(double2), what);
        if (!ok) set_error(QM_ERR_OUT_OF_MEMORY, "%s: %llu bytes of state memory", what, state_off * 16ULL);
    }
    if (ok) ok = dev_reserve((void**)&b->d_energies, &b->cap[2], std::max<size_t>(1, dc.size()) * sizeof(double), what);
    if (ok) ok = dev_reserve((void**)&b->d_partials, &b->cap[3], std::max<size_t>(1, nchunk) * sizeof(double), what);
    if (!ok) {
        b->release();
        return QM_ERR_HIP;
    }
    b->K = K;
    b->keep = keep_states ? 1 : 0;
    b->levels = levels;
    b->energy_items = energy_items;
    b->n_large = (u32)large.size();
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
    if (!b->lds_set && !batch_prepare_launch(b, what)) return nullptr;
    for (size_t lv = 0; lv < b->levels.size(); ++lv) {
        const qm_batch::Level& L = b->levels[lv];
        const size_t lds = sizeof(double2) << L.lq;
        const u32 groups = (1u << L.lq) >> b->K;
#define QM_BATCH_LEVEL(KK)                                                                                         \
    k_batch_level<KK><<<L.count, std::max(64u, std::min(tile_threads<KK>(), groups)), lds, st>>>(                  \
        b->d_circs, b->d_stages, b->d_passes, b->d_subs, b->d_pool, b->d_terms, b->d_items + L.first, (u32)lv,     \
        b->d_scratch, b->d_energies, b->keep)
        switch (b->K) {
            case 2: QM_BATCH_LEVEL(2); break;
            case 3: QM_BATCH_LEVEL(3); break;
            default: QM_BATCH_LEVEL(4); break;
        }
#undef QM_BATCH_LEVEL
    }
    if (b->n_large) {
        k_batch_energy<<<b->energy_items.count, kEnergyThreads, sizeof(double2) << kTileLocal, st>>>(b->d_circs, b->d_terms, b->d_items + b->energy_items.first,
                                                             b->d_scratch, b->d_partials);
        k_batch_finish<<<(b->n_large + 63) / 64, 64, 0, st>>>(b->d_circs, b->d_large, b->n_large, b->d_partials,
                                                              b->d_energies);
    }
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
    if (!b->lds_set && !batch_prepare_launch(b, what)) return QM_ERR_HIP;
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
    u32 K = block_qubits ? block_qubits : 3;
    u32 lq = local_qubits ? local_qubits : kTileLocal;
    if (n < kMinQubits || n > QM_CIRCUIT_MAX_QUBITS || K < 2 || K > 4 || lq < 8 || lq > kMaxLocal ||
        (gate_count && !gates)) {
        set_error(QM_ERR_INVALID_ARGUMENT,
                  "%s: need %u <= qubits (%u) <= %u, block_qubits (%u) in 2..4, local_qubits (%u) in 8..%u and a gate array",
                  what, kMinQubits, n, QM_CIRCUIT_MAX_QUBITS, K, lq, kMaxLocal);
        return nullptr;
    }
    auto* c = new qm_circuit();
    HCirc hc;
    if (!convert_gates(n, gates, gate_count, hc, what, true)) {
        delete c;
        return nullptr;
    }
    // blocks that hold the widest gate; depolarizing takes 4 (row and column bits of two qubits)
    auto needs = [](const HOp& o) { return o.type == 4 ? size_t(4) : o.type == 0 ? o.q.size() : size_t(0); };
    if (!block_qubits)  // the default width widens to the largest dense gate (at most 4 qubits)
        for (const HOp& o : hc.ops)
            if (needs(o) > K && needs(o) <= 4) K = (u32)needs(o);
    for (const HOp& o : hc.ops)
        if (needs(o) > K) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: a %zu-qubit dense gate needs block_qubits >= %zu", what, o.q.size(),
                      needs(o));
            delete c;
            return nullptr;
        }
    Flat f;
    schedule_circuit(f, hc, K, lq);
    // Defaults (0): 3-qubit blocks and 12-qubit windows (two work-groups per CU).  Against 4-qubit
    // blocks and 13-qubit windows (one per CU, prefetched), brickwork of 10 layers: 52 / 67 us
    // at 12 qubits, 83 / 116 at 16, 166 / 191 at 20, 405 / 398 at 22, 1377 / 1654 at 24,
    // 5.64 / 6.59 ms at 26; QAOA and random circuits alike.  The wider window pays where it saves a
    // stage, a pass over the state, of a circuit with little arithmetic, taken as two single-qubit
    // operations a qubit (a CNOT counts three, a matrix on k qubits 2^(k-1)).  Ten matrices between qubits 3 and 20: one stage instead of two, 46 / 31
    // us at 20 qubits, 210 / 169 at 24, 3.54 / 2.33 ms at 28; a layer of matrices and CZs at 22: two
    // instead of three, 118 / 114.  Without a stage saved it loses (that layer at 20: 46 / 57), and so it does
    // with more arithmetic (four CNOT ladders at 22 saving none 262 / 316, one at 23, three stages to
    // two, 230 / 250; 24 three-qubit unitaries on a 12-qubit density matrix 1.52 / 3.15 ms).  Below 20 qubits a state is some tens of tiles and stages cost the same.
    u64 work = 0;  // multiply-adds per amplitude, in those of a single-qubit matrix
    for (const HOp& o : hc.ops) work += o.type == 0 ? 1u << (o.q.size() - 1) : o.type == 4 ? o.q.size() : 1u;
    if (!block_qubits && !local_qubits && n >= 20 && work <= 2 * n) {
        Flat wide;
        schedule_circuit(wide, hc, 4, kMaxLocal);
        if (wide.stages.size() < f.stages.size()) {
            f = std::move(wide);
            K = 4;
            lq = kMaxLocal;
        }
    }
    c->n = n;
    c->K = K;
    c->lq = std::min(n, lq);
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
        auto round = [](size_t b) { return (b + 255) & ~size_t(255); };
        const size_t np = round(c->passes.size() * sizeof(DPass)), ns = round(c->subs.size() * sizeof(DSub));
        const size_t nm = c->pool.size() * sizeof(double2);
        std::vector<char> host(np + ns + nm);
        std::memcpy(host.data(), c->passes.data(), c->passes.size() * sizeof(DPass));
        std::memcpy(host.data() + np, c->subs.data(), c->subs.size() * sizeof(DSub));
        std::memcpy(host.data() + np + ns, c->pool.data(), nm);
        const char* what = "qm_circuit_apply: program";
        char* d = nullptr;
        if (!hip_ok(hipMalloc((void**)&d, host.size()), what)) return false;
        if (!hip_ok(hipMemcpy(d, host.data(), host.size(), hipMemcpyHostToDevice), what)) {
            (void)hipFree(d);
            return false;
        }
        c->d_program = d;
        c->d_passes = (DPass*)d;
        c->d_subs = (DSub*)(d + np);
        c->d_pool = (double2*)(d + np + ns);
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
    const u32 tl = c->n - c->lq;
    const u64 ntiles = 1ULL << tl;
    if (c->lq <= 12 && c->K >= 3) {
        const void* kt = c->K == 3 ? (const void*)k_tile<3> : (const void*)k_tile<4>;
        if (c->per_cu == 0) {
            if (!hip_ok(hipFuncSetAttribute(kt, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(double2) << 12)), what))
                return false;
            c->per_cu = 1;
        }
        // A thread per register block; a state of one tile takes full work-groups, whose other waves share
        // its loads, stores and the program's warm-up.  60 dense gates on four of 8 qubits: 379 -> 279 us.
        const u32 most = c->K == 3 ? tile_threads<3>() : tile_threads<4>();
        const u32 T = tl == 0 ? most : std::max(64u, std::min(most, (1u << c->lq) >> c->K));
        for (const DStage& sg : c->stages) {
            if (sg.npass == 0) continue;
            for (u64 t0 = 0; t0 < ntiles; t0 += kTilesPerLaunch) {
                const u32 nt = (u32)std::min<u64>(kTilesPerLaunch, ntiles - t0);
                if (c->K == 3) k_tile<3><<<nt, T, lds, st>>>((double2*)state, c->lq, tl, t0, sg, c->d_passes, c->d_subs, c->d_pool);
                else k_tile<4><<<nt, T, lds, st>>>((double2*)state, c->lq, tl, t0, sg, c->d_passes, c->d_subs, c->d_pool);
            }
        }
        return hip_ok(hipGetLastError(), what);
    }
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
