// Reductions over a state vector, in FP64, deterministic: every block reduces
// a fixed slice (wave shuffle tree, then a fixed-order sum over waves) into a
// partials array, and one block sums the partials in index order.  No atomics,
// no per-call allocation (the reference allocates, memsets and atomically adds
// per call: src/gpusim/stat_ops.cu:140-198).
//
// Reference loops restated: src/csim/stat_ops.cpp:13-86,
// stat_ops_probability.cpp:11-100, stat_ops_expectation_value.cpp:352-482,
// stat_ops_transition_amplitude.cpp:19-128, update_ops_named_state.cpp:21-98.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "qm_internal.hpp"

namespace qm {

constexpr int kRBlock = 256;
constexpr unsigned kMaxRBlocks = 2048;

// real part of z * i^k
__device__ __forceinline__ double re_rot(double2 z, unsigned k) {
    switch (k & 3) {
        case 0: return z.x;
        case 1: return -z.y;
        case 2: return -z.x;
        default: return z.y;
    }
}
__device__ __forceinline__ double2 rot(double2 z, unsigned k) {  // z * i^k
    switch (k & 3) {
        case 0: return z;
        case 1: return make_double2(-z.y, z.x);
        case 2: return make_double2(-z.x, -z.y);
        default: return make_double2(z.y, -z.x);
    }
}
__device__ __forceinline__ unsigned par(u64 x) { return __popcll(x) & 1; }
__device__ __forceinline__ double norm2(double2 v) { return fma(v.x, v.x, v.y * v.y); }

// One Pauli term (or a plain reduction) as seen by the kernels.
struct Term {
    u64 bf, pf;
    unsigned rot, pivot;
};

// Kinds of per-element functionals.
enum RKind : int {
    R_NORM = 0,      // sum |psi_i|^2
    R_ENTROPY = 1,   // sum -p log p with p clamped to >= 1e-15
    R_MASKED = 2,    // sum |psi_b|^2 over b with (b & mask) == value (M0, M1, marginal)
    R_PAULI = 3,     // <psi|P|psi> (XZ or Z form per term)
    R_TRANS = 4,     // <bra|P|ket> (complex)
    R_INNER = 5,     // <bra|ket> (complex)
};

struct RArgs {
    const double2* __restrict__ a;  // state / ket
    const double2* __restrict__ b;  // bra (R_TRANS, R_INNER)
    u64 dim;
    u64 mask, value;                // R_MASKED
    Term term;                      // R_PAULI / R_TRANS
    double* __restrict__ partials;  // [gridDim.y][gridDim.x][2]
    double* __restrict__ out;       // a grid of one block: its result goes here, and nothing follows
};

template <int KIND>
__global__ __launch_bounds__(kRBlock) void k_reduce(RArgs r) {
    __shared__ double lds[32];
    double acc_re = 0.0, acc_im = 0.0;
    const u64 stride = (u64)gridDim.x * blockDim.x;
    const u64 t0 = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (KIND == R_NORM) {
        for (u64 i = t0; i < r.dim; i += stride) acc_re += norm2(r.a[i]);
    } else if (KIND == R_ENTROPY) {
        for (u64 i = t0; i < r.dim; i += stride) {
            double p = norm2(r.a[i]);
            p = p > 1e-15 ? p : 1e-15;
            acc_re += -p * log(p);
        }
    } else if (KIND == R_MASKED) {
        for (u64 i = t0; i < r.dim; i += stride)
            if ((i & r.mask) == r.value) acc_re += norm2(r.a[i]);
    } else if (KIND == R_PAULI) {
        const Term tm = r.term;
        if (tm.bf == 0) {
            for (u64 i = t0; i < r.dim; i += stride) {
                const double p = norm2(r.a[i]);
                acc_re += par(i & tm.pf) ? -p : p;
            }
        } else {
            const u64 half = r.dim >> 1;
            for (u64 i = t0; i < half; i += stride) {
                const u64 b0 = insert_zero(i, tm.pivot), b1 = b0 ^ tm.bf;
                const double2 x = r.a[b0], y = r.a[b1];
                // x * conj(y)
                const double2 z = make_double2(fma(x.x, y.x, x.y * y.y), fma(x.y, y.x, -x.x * y.y));
                acc_re += 2.0 * re_rot(z, tm.rot + 2 * par(b0 & tm.pf));
            }
        }
    } else if (KIND == R_TRANS) {
        const Term tm = r.term;
        const double2* ket = r.a;
        const double2* bra = r.b;
        if (tm.bf == 0) {
            for (u64 i = t0; i < r.dim; i += stride) {
                const double2 k = ket[i], b = bra[i];
                // k * conj(b)
                double2 z = make_double2(fma(k.x, b.x, k.y * b.y), fma(k.y, b.x, -k.x * b.y));
                if (par(i & tm.pf)) z = make_double2(-z.x, -z.y);
                acc_re += z.x;
                acc_im += z.y;
            }
        } else {
            const u64 half = r.dim >> 1;
            for (u64 i = t0; i < half; i += stride) {
                const u64 b0 = insert_zero(i, tm.pivot), b1 = b0 ^ tm.bf;
                const double2 k0 = ket[b0], k1 = ket[b1], c0 = bra[b0], c1 = bra[b1];
                const double2 z1 = rot(make_double2(fma(k0.x, c1.x, k0.y * c1.y), fma(k0.y, c1.x, -k0.x * c1.y)),
                                       tm.rot + 2 * par(b0 & tm.pf));
                const double2 z2 = rot(make_double2(fma(k1.x, c0.x, k1.y * c0.y), fma(k1.y, c0.x, -k1.x * c0.y)),
                                       tm.rot + 2 * par(b1 & tm.pf));
                acc_re += z1.x + z2.x;
                acc_im += z1.y + z2.y;
            }
        }
    } else if (KIND == R_INNER) {
        for (u64 i = t0; i < r.dim; i += stride) {
            const double2 b = r.b[i], k = r.a[i];
            // conj(b) * k
            acc_re += fma(b.x, k.x, b.y * k.y);
            acc_im += fma(b.x, k.y, -b.y * k.x);
        }
    }
    const double s_re = block_sum(acc_re, lds);
    double s_im = 0.0;
    if (KIND == R_TRANS || KIND == R_INNER) s_im = block_sum(acc_im, lds);
    if (threadIdx.x == 0) {
        double* out = r.out ? r.out : r.partials + ((u64)blockIdx.y * gridDim.x + blockIdx.x) * 2;
        out[0] = s_re;
        out[1] = s_im;
    }
}

// Sums `count` (re, im) pairs of partials in a fixed order (thread-strided, then a fixed tree)
// into out, which may be pinned host memory: a copy command for 16 bytes costs more than the
// kernel.  add: onto what an earlier launch of the stream left there.
constexpr int kFinishThreads = 256;
__global__ __launch_bounds__(kFinishThreads) void k_finish(const double* __restrict__ partials, unsigned count,
                                                           double* __restrict__ out, bool add = false) {
    __shared__ double lds[32];
    double re = 0.0, im = 0.0;
    for (unsigned k = threadIdx.x; k < count; k += kFinishThreads) {
        re += partials[2 * k];
        im += partials[2 * k + 1];
    }
    re = block_sum(re, lds);
    im = block_sum(im, lds);
    if (threadIdx.x == 0) {
        out[0] = add ? out[0] + re : re;
        out[1] = add ? out[1] + im : im;
    }
}

unsigned reduce_blocks(u64 work) { return grid_for(work, (u64)kRBlock * 16, kMaxRBlocks); }

// Runs one reduction and waits for it; `term` for R_PAULI and R_TRANS.  Returns false on error;
// the result (re, im) in res.
template <int KIND>
bool run_reduce(RArgs r, u64 work, const Term* term, hipStream_t st, double res[2]) {
    Scratch* sc = scratch_for(st);
    if (!sc) return false;
    const unsigned nb = reduce_blocks(work);
    if (term) r.term = *term;
    r.partials = sc->partials;
    r.out = nb == 1 ? sc->host_result : nullptr;
    k_reduce<KIND><<<nb, kRBlock, 0, st>>>(r);
    if (nb > 1) k_finish<<<1, kFinishThreads, 0, st>>>(sc->partials, nb, sc->host_result);
    if (!hip_ok(hipGetLastError(), "reduce") || !hip_ok(hipStreamSynchronize(st), "reduce sync")) return false;
    res[0] = sc->host_result[0];
    res[1] = sc->host_result[1];
    return true;
}

// ------------------------------------------------------------------ observables
// sum_k c_k <psi|P_k|psi>.  A term with bit-flip mask bf pairs index x with x ^ bf, so one pass
// per term reads the whole state for one number.  Terms are put into groups whose masks span at
// most 4 dimensions over GF(2): the 16 amplitudes of a coset of the span meet only each other
// in all of a group's terms, so a thread loads one coset and evaluates them all, and the state
// is read once per group.  With the span in reduced echelon form (pivot bits p_0..p_3), cosets
// are numbered by the index bits that are no pivots, and member m is base ^ (sum of the
// basis vectors in m); a term is the pairs (m, m ^ e), e = its mask's pivot bits, with the
// sign (-1)^popcount(index & pf) = (lane: base & pf) x (uniform: bit m of a 16-bit pattern).
// Bound: HBM.  25 qubits, 24 random terms: 24 passes, 1.91 ms; with 6 groups 0.51 ms (6.3 TB/s).
constexpr int kObsRank = 4;
constexpr int kObsMembers = 1 << kObsRank;
constexpr unsigned kObsInlineTerms = 48, kObsInlineGroups = 16;  // passed as kernel arguments
constexpr unsigned kObsMaxBlocks = 2048, kObsMaxGroups = 256;   // per launch: the partials hold this many pairs
constexpr unsigned kObsMaxTerms = 1u << 16;                      // of a call that does not wait: the upload ring takes their tables
constexpr u64 kObsOneBlock = 1ULL << 13;  // states up to here may take one block
constexpr u64 kObsOneTerms = 8;           // terms, times cosets of a thread, per wave or block of that launch
constexpr unsigned kObsSpread = 1024;     // work-groups that a launch of many terms is spread over
constexpr u64 kObsByWave = 64 * kObsMembers;  // states up to here: a group per wave

struct ObsTerm {
    u64 bf, pf;
    u32 e, pattern;   // e: pairs (m, m ^ e), odd: 16 set if the imaginary part counts
    double cre, cim;  // coefficient with the factor 2 of a pair and the sign of i^rot
};
struct ObsGroup {
    u64 basis[kObsRank];
    u32 term0, nterm;
    unsigned char piv[kObsRank];  // ascending
    u32 pad;
};
struct ObsArgs {
    const double2* state;
    u64 dim;
    double* partials;  // [group][gridDim.x][2]
    double* out;       // a single block writes the total here
    u32 ngroup;
    const ObsTerm* terms;    // more than the arrays below hold
    const ObsGroup* groups;
    ObsTerm term[kObsInlineTerms];
    ObsGroup group[kObsInlineGroups];
};

template <int E, bool ODD>
__device__ __forceinline__ double pair_sum(const double2 (&v)[kObsMembers], u32 pattern) {
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < kObsMembers; ++m) {
        if (m > (m ^ E)) continue;
        const double2 a = v[m], b = v[m ^ E];
        const double t = ODD ? fma(a.y, b.x, -a.x * b.y) : fma(a.x, b.x, a.y * b.y);
        s = fma(t, ((pattern >> m) & 1u) ? -1.0 : 1.0, s);
    }
    return s;
}
__device__ __forceinline__ double term_sum(const double2 (&v)[kObsMembers], u32 e, u32 pattern) {
    switch (e) {
#define QM_OBS_CASE(E)                                     \
    case E: return pair_sum<E, false>(v, pattern);         \
    case E + 16: return pair_sum<E, true>(v, pattern);
        QM_OBS_CASE(1) QM_OBS_CASE(2) QM_OBS_CASE(3) QM_OBS_CASE(4) QM_OBS_CASE(5) QM_OBS_CASE(6) QM_OBS_CASE(7)
        QM_OBS_CASE(8) QM_OBS_CASE(9) QM_OBS_CASE(10) QM_OBS_CASE(11) QM_OBS_CASE(12) QM_OBS_CASE(13) QM_OBS_CASE(14)
        QM_OBS_CASE(15)
#undef QM_OBS_CASE
        default: return pair_sum<0, false>(v, pattern);
    }
}

template <bool INLINE>
__global__ __launch_bounds__(kRBlock) void k_observable(ObsArgs a) {
    __shared__ double lds[32];
    double re = 0.0, im = 0.0;
    // up to 64 cosets: a group per wave instead of the groups one after another
    const bool by_wave = a.dim <= kObsByWave;
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const u64 stride = by_wave ? 64 : (u64)gridDim.x * blockDim.x;
    const u64 t0 = by_wave ? threadIdx.x & 63 : (u64)blockIdx.x * blockDim.x + threadIdx.x;
    const double2* __restrict__ psi = a.state;
    const u32 side = by_wave ? kRBlock / 64 : 1;  // groups side by side in a block
    for (u32 g = blockIdx.y * side + (by_wave ? wave : 0); g < a.ngroup; g += gridDim.y * side) {
        const ObsGroup gr = INLINE ? a.group[g] : a.groups[g];
        if (a.dim < (u64)kObsMembers) {  // fewer amplitudes than a coset has
            if (t0 < a.dim) {
                for (u32 k = 0; k < gr.nterm; ++k) {
                    const ObsTerm tm = INLINE ? a.term[gr.term0 + k] : a.terms[gr.term0 + k];
                    const double2 x = psi[t0], y = psi[t0 ^ tm.bf];
                    double t = (tm.e & 16u) ? fma(x.y, y.x, -x.x * y.y) : fma(x.x, y.x, x.y * y.y);
                    if (tm.bf) t *= 0.5;  // every pair is met from both sides
                    if (par(t0 & tm.pf)) t = -t;
                    re = fma(tm.cre, t, re);
                    im = fma(tm.cim, t, im);
                }
            }
            continue;
        }
        for (u64 i = t0; i < a.dim / kObsMembers; i += stride) {
            u64 base = i;
#pragma unroll
            for (int k = 0; k < kObsRank; ++k) base = insert_zero(base, gr.piv[k]);
            double2 v[kObsMembers];
#pragma unroll
            for (int m = 0; m < kObsMembers; ++m) {
                const u64 off = ((m & 1) ? gr.basis[0] : 0) ^ ((m & 2) ? gr.basis[1] : 0) ^ ((m & 4) ? gr.basis[2] : 0) ^
                                ((m & 8) ? gr.basis[3] : 0);
                v[m] = psi[base ^ off];
            }
            for (u32 k = 0; k < gr.nterm; ++k) {
                const ObsTerm tm = INLINE ? a.term[gr.term0 + k] : a.terms[gr.term0 + k];
                // keeps the products of all 31 cases from being formed in front of the loop
#pragma unroll
                for (int m = 0; m < kObsMembers; ++m) asm volatile("" : "+v"(v[m].x), "+v"(v[m].y));
                double t = term_sum(v, tm.e, tm.pattern);
                if (par(base & tm.pf)) t = -t;
                re = fma(tm.cre, t, re);
                im = fma(tm.cim, t, im);
            }
        }
    }
    re = block_sum(re, lds);
    im = block_sum(im, lds);
    if (threadIdx.x == 0) {
        double* out = a.out ? a.out : a.partials + ((u64)blockIdx.y * gridDim.x + blockIdx.x) * 2;
        out[0] = re;
        out[1] = im;
    }
}

// Groups the terms of an observable on n qubits.
struct ObsPlan {
    std::vector<ObsTerm> terms;  // group after group
    std::vector<ObsGroup> groups;
    unsigned nb = 1;       // blocks along the state
    bool by_wave = false;  // small states: see k_observable
    bool one = false;      // one block does all
    // blocks along the groups for ng of them
    unsigned ny(size_t ng) const { return one ? 1u : (unsigned)(by_wave ? (ng + 3) / 4 : ng); }
    // groups of a launch whose partials fit (2^20 doubles)
    size_t per_launch() const { return std::min<size_t>(1u << 15, (size_t)kObsMaxBlocks * kObsMaxGroups / nb); }
};
// The grid.  One block for a small state and few terms needs no second launch; its waves wait
// out the latency of one term after another (0.4 us each), so it takes kObsOneTerms of them.  Beyond
// that, and on larger states with few blocks and groups (all Z strings are one group), groups are
// split until some kObsSpread blocks share the terms: their pieces read the same state, from L2.
// 12 random terms at 12 qubits: one block 22.8 us, spread 20.4; 4 terms at 13 qubits 19.0 and 20.0.
// 1000 terms at 13 qubits: one block 1150 us, spread 130; 1000 Z strings at 16: one group 481, spread 78.
void shape_observable(ObsPlan& pl, u64 dim) {
    const u64 cosets = std::max<u64>(1, dim / kObsMembers), terms = pl.terms.size();
    pl.by_wave = dim <= kObsByWave;
    pl.nb = pl.by_wave ? 1u : (unsigned)std::min<u64>(kObsMaxBlocks, (cosets + kRBlock - 1) / kRBlock);
    const u64 side = pl.by_wave ? 4 : 1;
    pl.one = dim <= kObsOneBlock && terms * pl.nb <= kObsOneTerms * side;
    u64 piece = terms;
    if (pl.one) {
        pl.nb = 1;
        if (pl.by_wave && pl.groups.size() < side) piece = std::max<u64>(4, (terms + side - 1) / side);
    } else {
        piece = std::max<u64>(8, (terms * pl.nb + kObsSpread * side - 1) / (kObsSpread * side));
    }
    std::vector<ObsGroup> out;
    for (const ObsGroup& g : pl.groups)
        for (u32 t = 0; t < g.nterm; t += (u32)piece) {
            out.push_back(g);
            out.back().term0 = g.term0 + t;
            out.back().nterm = std::min<u32>((u32)piece, g.nterm - t);
        }
    // (not where the groups alone are kernel arguments: an upload costs more than it saves)
    if (terms > kObsInlineTerms || out.size() <= kObsInlineGroups || pl.groups.size() > kObsInlineGroups)
        pl.groups.swap(out);
}
ObsPlan plan_observable(const u64* bf, const u64* pf, const u32* rot, const qm_complex* coef, u32 nterms, int n) {
    ObsPlan pl;
    // the distinct flip masks, by their highest bit, dealt out so that the pivots of a group are
    // spread over the register: low pivots alone would make a wave's loads touch 16-byte pieces
    // of distant lines
    std::vector<u64> masks;
    for (u32 k = 0; k < nterms; ++k)
        if (bf[k]) masks.push_back(bf[k]);
    std::sort(masks.begin(), masks.end());
    masks.erase(std::unique(masks.begin(), masks.end()), masks.end());
    const size_t D = masks.size(), deal = std::max<size_t>(1, (D + kObsRank - 1) / kObsRank);
    std::vector<u64> order;
    for (size_t g = 0; g < deal; ++g)
        for (size_t k = g; k < D; k += deal) order.push_back(masks[k]);
    struct Space {
        std::vector<u64> basis;  // reduced echelon form, pivot = highest bit of each
        u64 reduce(u64 v) const {
            for (u64 b : basis)
                if ((v >> (63 - __builtin_clzll(b))) & 1) v ^= b;
            return v;
        }
        void insert(u64 v) {  // v reduced and not 0
            const int p = 63 - __builtin_clzll(v);
            for (u64& b : basis)
                if ((b >> p) & 1) b ^= v;
            basis.push_back(v);
        }
    };
    std::vector<Space> spaces(1);
    // group of each mask (sorted); a mask in an earlier group's span joins it (searched
    // while there are few)
    std::vector<u32> group_of(D, 0);
    auto index_of = [&](u64 m) { return (size_t)(std::lower_bound(masks.begin(), masks.end(), m) - masks.begin()); };
    for (u64 m : order) {
        size_t g = spaces.size() - 1;
        bool found = false;
        for (size_t k = D <= 256 ? 0 : g; k <= g && !found; ++k)
            if (spaces[k].reduce(m) == 0) {
                group_of[index_of(m)] = (u32)k;
                found = true;
            }
        if (found) continue;
        if (spaces[g].basis.size() == (size_t)kObsRank || (int)spaces[g].basis.size() == n) {
            spaces.emplace_back();
            ++g;
        }
        spaces[g].insert(spaces[g].reduce(m));
        group_of[index_of(m)] = (u32)g;
    }
    // fill every basis up to the full rank with single high bits
    for (Space& sp : spaces)
        for (int q = n - 1; q >= 0 && sp.basis.size() < (size_t)kObsRank; --q)
            if (sp.reduce(1ULL << q)) sp.insert(sp.reduce(1ULL << q));
    std::vector<std::vector<u32>> members(spaces.size());
    for (u32 k = 0; k < nterms; ++k) members[bf[k] ? group_of[index_of(bf[k])] : 0].push_back(k);
    for (size_t g = 0; g < spaces.size(); ++g) {
        std::vector<u64>& b = spaces[g].basis;
        std::sort(b.begin(), b.end());  // ascending pivots
        ObsGroup gr{};
        for (size_t k = 0; k < b.size(); ++k) {
            gr.basis[k] = b[k];
            gr.piv[k] = (unsigned char)(63 - __builtin_clzll(b[k]));
        }
        gr.term0 = (u32)pl.terms.size();
        gr.nterm = (u32)members[g].size();
        for (u32 k : members[g]) {
            ObsTerm t{};
            t.bf = bf[k];
            t.pf = pf[k];
            for (size_t i = 0; i < b.size(); ++i) t.e |= (u32)((bf[k] >> gr.piv[i]) & 1u) << i;
            for (u32 m = 0; m < (u32)kObsMembers; ++m) {
                u64 off = 0;
                for (size_t i = 0; i < b.size(); ++i)
                    if ((m >> i) & 1) off ^= b[i];
                t.pattern |= (u32)(__builtin_popcountll(off & pf[k]) & 1) << m;
            }
            // a pair gives 2 Re(z i^rot), z = psi_x conj(psi_y) and x's parity; a Z string |psi_x|^2
            double f = 1.0;
            if (bf[k]) {
                const u32 r = rot[k] & 3u;
                f = (r == 1 || r == 2) ? -2.0 : 2.0;
                if (r & 1u) t.e |= 16u;
            }
            t.cre = f * coef[k].re;
            t.cim = f * coef[k].im;
            pl.terms.push_back(t);
        }
        pl.groups.push_back(gr);
    }
    shape_observable(pl, 1ULL << n);
    return pl;
}

// Enqueues the groups [g0, g0 + ng) of a plan; their sum goes to out (device or pinned memory),
// added to what is there if `add`.
// dterms and dgroups hold the terms and groups in device memory when they are too many for the arguments.
bool launch_observable(const ObsPlan& pl, size_t g0, size_t ng, const void* state, u64 dim, hipStream_t st,
                       double* partials, const ObsTerm* dterms, const ObsGroup* dgroups, double* out, const char* what,
                       bool add = false) {
    ObsArgs a{};
    a.state = (const double2*)state;
    a.dim = dim;
    a.partials = partials;
    a.ngroup = (u32)ng;
    a.terms = dterms;
    a.groups = dgroups ? dgroups + g0 : nullptr;
    const unsigned nb = pl.nb, ny = pl.ny(ng);
    a.out = nb * ny == 1 && !add ? out : nullptr;
    if (!dterms) {
        std::copy(pl.terms.begin(), pl.terms.end(), a.term);
        std::copy(pl.groups.begin(), pl.groups.end(), a.group);
        k_observable<true><<<dim3(nb, ny), kRBlock, 0, st>>>(a);
    } else {
        k_observable<false><<<dim3(nb, ny), kRBlock, 0, st>>>(a);
    }
    if (!a.out) k_finish<<<1, kFinishThreads, 0, st>>>(partials, nb * ny, out, add);
    return hip_ok(hipGetLastError(), what);
}
bool obs_inline(const ObsPlan& pl) {
    return pl.terms.size() <= kObsInlineTerms && pl.groups.size() <= kObsInlineGroups;
}

// The tables of a plan that the kernel arguments do not hold, in one copy.
bool upload_plan(Scratch* sc, const ObsPlan& pl, const ObsTerm** dterms, const ObsGroup** dgroups) {
    const size_t nt = pl.terms.size() * sizeof(ObsTerm), ng = pl.groups.size() * sizeof(ObsGroup);
    std::vector<char> host(nt + ng);
    std::memcpy(host.data(), pl.terms.data(), nt);
    std::memcpy(host.data() + nt, pl.groups.data(), ng);
    const char* d = (const char*)upload(sc, host.data(), host.size());
    if (!d) return false;
    *dterms = (const ObsTerm*)d;
    *dgroups = (const ObsGroup*)(d + nt);
    return true;
}
static_assert(kObsMaxTerms * (sizeof(ObsTerm) + sizeof(ObsGroup)) <= kRingBytes, "the ring takes a plan's tables");

bool enqueue_observable(const u64* bf, const u64* pf, const u32* rot, const double* coef, u32 nterms,
                        const void* state, u64 dim, hipStream_t st, double* h_out) {
    const char* what = "enqueue_observable";
    h_out[0] = h_out[1] = 0.0;
    if (nterms == 0) return true;
    if (nterms > kObsMaxTerms) {
        set_error(QM_ERR_UNSUPPORTED, "%s: too many terms in one observable (%u)", what, nterms);
        return false;
    }
    std::vector<qm_complex> c(nterms);
    for (u32 k = 0; k < nterms; ++k) c[k] = qm_complex{coef[k], 0.0};
    const ObsPlan pl = plan_observable(bf, pf, rot, c.data(), nterms, log2_dim(dim));
    Scratch* sc = scratch_for(st);
    if (!sc) return false;
    const ObsTerm* dt = nullptr;
    const ObsGroup* dg = nullptr;
    if (!obs_inline(pl) && !upload_plan(sc, pl, &dt, &dg)) return false;
    for (size_t g = 0; g < pl.groups.size(); g += pl.per_launch())
        if (!launch_observable(pl, g, std::min(pl.per_launch(), pl.groups.size() - g), state, dim, st, sc->partials,
                               dt, dg, h_out, what, g > 0))
            return false;
    return true;
}

bool state_ok(const void* s, u64 dim, const char* what) {
    if (!s || log2_dim(dim) < 0) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null state or dim %llu is not a power of two >= 2", what, dim);
        return false;
    }
    return true;
}

Term make_term(u64 bf, u64 pf, unsigned rot, unsigned pivot) {
    Term t;
    t.bf = bf;
    t.pf = pf;
    t.rot = rot & 3;
    t.pivot = pivot;
    return t;
}

bool pauli_term_from_list(const u32* tl, const u32* pl, u32 n, int nq, Term* t, const char* what) {
    u64 bf = 0, pf = 0;
    unsigned rot = 0, pivot = 0;
    for (u32 c = 0; c < n; ++c) {
        if ((int)tl[c] >= nq) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: qubit %u out of range", what, tl[c]);
            return false;
        }
        switch (pl[c]) {
            case 0: break;
            case 1: bf ^= 1ULL << tl[c]; pivot = tl[c]; break;
            case 2: bf ^= 1ULL << tl[c]; pf ^= 1ULL << tl[c]; rot++; pivot = tl[c]; break;
            case 3: pf ^= 1ULL << tl[c]; break;
            default:
                set_error(QM_ERR_INVALID_ARGUMENT, "%s: Pauli id %u out of 0..3", what, pl[c]);
                return false;
        }
    }
    *t = make_term(bf, pf, rot, pivot);
    return true;
}

double pauli_expectation(const Term& t, void* state, u64 dim, void* stream, unsigned dev, const char* what) {
    if (!state_ok(state, dim, what)) return 0.0;
    const int n = log2_dim(dim);
    if (((t.bf | t.pf) >> n) != 0 || (t.bf && !((t.bf >> t.pivot) & 1))) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: masks beyond %d qubits or pivot outside the flip mask", what, n);
        return 0.0;
    }
    if (!use_device(dev)) return 0.0;
    RArgs r{};
    r.a = (const double2*)state;
    r.dim = dim;
    double res[2] = {0, 0};
    run_reduce<R_PAULI>(r, t.bf ? dim / 2 : dim, &t, stream_of(stream), res);
    return res[0];
}

qm_complex transition(const Term& t, void* bra, void* ket, u64 dim, void* stream, unsigned dev, const char* what) {
    qm_complex z{0, 0};
    if (!state_ok(bra, dim, what) || !state_ok(ket, dim, what)) return z;
    const int n = log2_dim(dim);
    if (((t.bf | t.pf) >> n) != 0 || (t.bf && !((t.bf >> t.pivot) & 1))) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: masks beyond %d qubits or pivot outside the flip mask", what, n);
        return z;
    }
    if (!use_device(dev)) return z;
    RArgs r{};
    r.a = (const double2*)ket;
    r.b = (const double2*)bra;
    r.dim = dim;
    double res[2] = {0, 0};
    if (run_reduce<R_TRANS>(r, t.bf ? dim / 2 : dim, &t, stream_of(stream), res)) {
        z.re = res[0];
        z.im = res[1];
    }
    return z;
}

// ------------------------------------------------------------------ elementwise state arithmetic
__global__ __launch_bounds__(256) void k_axpy(double2* __restrict__ s, const double2* __restrict__ a, u64 dim,
                                              double2 coef) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) st_stream(s + i, cmac(ld_stream(s + i), coef, ld_stream(a + i)));
}
__global__ __launch_bounds__(256) void k_add(double2* __restrict__ s, const double2* __restrict__ a, u64 dim) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) st_stream(s + i, cadd(ld_stream(s + i), ld_stream(a + i)));
}
// Elementwise in-place passes: from 128 amplitudes up, each thread takes two
// amplitudes 64 apart (both loads issued before either store), so a wave reads
// 2 KiB of consecutive lines per iteration; smaller states take one per thread.
template <class F>
__device__ __forceinline__ void inplace_pass(double2* __restrict__ s, u64 dim, F f) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    const u64 t0 = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (dim < 128) {
        for (u64 i = t0; i < dim; i += stride) s[i] = f(s[i]);
        return;
    }
    for (u64 i = t0; i < (dim >> 1); i += stride) {
        const u64 a = ((i >> 6) << 7) | (i & 63);
        const double2 x = ld_stream(s + a), y = ld_stream(s + a + 64);
        st_stream(s + a, f(x));
        st_stream(s + a + 64, f(y));
    }
}
__global__ __launch_bounds__(512) void k_scale_c(double2* __restrict__ s, u64 dim, double2 coef) {
    inplace_pass(s, dim, [coef](double2 v) { return cmul(v, coef); });
}
__global__ __launch_bounds__(512) void k_scale_r(double2* __restrict__ s, u64 dim, double f) {
    inplace_pass(s, dim, [f](double2 v) { return cscale(v, f); });
}

// ------------------------------------------------------------------ allocation-free observable
// qm_observable_expectation_noalloc_host runs the same launches as
// qm_observable_expectation_host (k_observable, then k_finish), but its tables, per-block
// partials and results live in `scratch`, a fixed device array, instead of the library's
// per-stream allocations.  Every block writes its partial slot and k_finish writes the result,
// so nothing in it has to start at zero.  All calls on one device share that device's copy: calls
// that overlap on one device (other threads, other streams) race.
constexpr unsigned kNoAllocMaxTerms = 128;
constexpr size_t kNoAllocTermsOff = 0;
constexpr size_t kNoAllocGroupsOff = 6144;    // >= 128 * sizeof(ObsTerm)
constexpr size_t kNoAllocOutOff = 14336;      // >= kNoAllocGroupsOff + 128 * sizeof(ObsGroup)
constexpr size_t kNoAllocPartialsOff = 14592;
constexpr size_t kNoAllocBytes = kNoAllocPartialsOff + (size_t)kObsMaxBlocks * kNoAllocMaxTerms * 2 * sizeof(double);
static_assert(kNoAllocMaxTerms * sizeof(ObsTerm) <= kNoAllocGroupsOff, "term table overlaps the groups");
static_assert(kNoAllocGroupsOff + kNoAllocMaxTerms * sizeof(ObsGroup) <= kNoAllocOutOff, "groups overlap the result");
static_assert(kNoAllocPartialsOff % 256 == 0, "partials not 256-byte aligned");

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
unsigned char* g_noalloc_ptr[kNoAllocMaxDevices] = {};

// Device address of `scratch` on the current device (looked up once per
// device; the array's name itself is only a host-side stand-in).
unsigned char* noalloc_scratch(unsigned dev, const char* what) {
    if (dev >= (unsigned)kNoAllocMaxDevices) {
        set_error(QM_ERR_UNSUPPORTED, "%s: device %u beyond %d", what, dev, kNoAllocMaxDevices);
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void* p = nullptr;
        if (!hip_ok(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), what)) return nullptr;
        g_noalloc_ptr[dev] = (unsigned char*)p;
    }
    return g_noalloc_ptr[dev];
}

}  // namespace qm

using namespace qm;

extern "C" {

double state_norm_squared_host(void* state, ITYPE dim, void* stream, unsigned dev) {
    if (!state_ok(state, dim, "state_norm_squared_host") || !use_device(dev)) return 0.0;
    RArgs r{};
    r.a = (const double2*)state;
    r.dim = dim;
    double res[2] = {0, 0};
    run_reduce<R_NORM>(r, dim, nullptr, stream_of(stream), res);
    return res[0];
}

double state_norm_squared_cublas_host(void* state, ITYPE dim) {
    return state_norm_squared_host(state, dim, nullptr, (unsigned)get_current_device());
}

double measurement_distribution_entropy_host(void* state, ITYPE dim, void* stream, unsigned dev) {
    if (!state_ok(state, dim, "measurement_distribution_entropy_host") || !use_device(dev)) return 0.0;
    RArgs r{};
    r.a = (const double2*)state;
    r.dim = dim;
    double res[2] = {0, 0};
    run_reduce<R_ENTROPY>(r, dim, nullptr, stream_of(stream), res);
    return res[0];
}

static double masked_prob(u64 mask, u64 value, void* state, ITYPE dim, void* stream, unsigned dev, const char* what) {
    if (!state_ok(state, dim, what) || !use_device(dev)) return 0.0;
    RArgs r{};
    r.a = (const double2*)state;
    r.dim = dim;
    r.mask = mask;
    r.value = value;
    double res[2] = {0, 0};
    run_reduce<R_MASKED>(r, dim, nullptr, stream_of(stream), res);
    return res[0];
}

double M0_prob_host(UINT t, void* state, ITYPE dim, void* stream, unsigned dev) {
    QM_CHECK_ARG_RET(log2_dim(dim) > (int)t, 0.0, "M0_prob_host: qubit %u out of range", t);
    return masked_prob(1ULL << t, 0, state, dim, stream, dev, "M0_prob_host");
}
double M1_prob_host(UINT t, void* state, ITYPE dim, void* stream, unsigned dev) {
    QM_CHECK_ARG_RET(log2_dim(dim) > (int)t, 0.0, "M1_prob_host: qubit %u out of range", t);
    return masked_prob(1ULL << t, 1ULL << t, state, dim, stream, dev, "M1_prob_host");
}
double marginal_prob_host(UINT* tl, UINT* vl, UINT n, void* state, ITYPE dim, void* stream, unsigned dev) {
    const int nq = log2_dim(dim);
    u64 mask = 0, value = 0;
    for (UINT i = 0; i < n; ++i) {
        QM_CHECK_ARG_RET((int)tl[i] < nq && vl[i] <= 1 && !((mask >> tl[i]) & 1), 0.0,
                         "marginal_prob_host: bad qubit %u / value %u", tl[i], vl[i]);
        mask |= 1ULL << tl[i];
        value |= (u64)vl[i] << tl[i];
    }
    return masked_prob(mask, value, state, dim, stream, dev, "marginal_prob_host");
}

double expectation_value_multi_qubit_Pauli_operator_XZ_mask_host(ITYPE bf, ITYPE pf, UINT rot, UINT pivot,
                                                                 void* state, ITYPE dim, void* stream, unsigned dev) {
    QM_CHECK_ARG_RET(bf != 0, 0.0, "expectation XZ mask: empty bit-flip mask");
    return pauli_expectation(make_term(bf, pf, rot, pivot), state, dim, stream, dev,
                             "expectation_value_multi_qubit_Pauli_operator_XZ_mask_host");
}
double expectation_value_multi_qubit_Pauli_operator_Z_mask_host(ITYPE pf, void* state, ITYPE dim, void* stream,
                                                                unsigned dev) {
    return pauli_expectation(make_term(0, pf, 0, 0), state, dim, stream, dev,
                             "expectation_value_multi_qubit_Pauli_operator_Z_mask_host");
}
double expectation_value_multi_qubit_Pauli_operator_partial_list_host(const UINT* tl, const UINT* pl, UINT n,
                                                                      void* state, ITYPE dim, void* stream,
                                                                      unsigned dev) {
    const char* what = "expectation_value_multi_qubit_Pauli_operator_partial_list_host";
    if (!state_ok(state, dim, what)) return 0.0;
    Term t;
    if (!pauli_term_from_list(tl, pl, n, log2_dim(dim), &t, what)) return 0.0;
    return pauli_expectation(t, state, dim, stream, dev, what);
}
double expectation_value_multi_qubit_Pauli_operator_whole_list_host(const UINT* pl, UINT n, void* state, ITYPE dim,
                                                                    void* stream, unsigned dev) {
    std::vector<u32> tl(n);
    for (UINT i = 0; i < n; ++i) tl[i] = i;
    return expectation_value_multi_qubit_Pauli_operator_partial_list_host(tl.data(), pl, n, state, dim, stream, dev);
}
double expectation_value_single_qubit_Pauli_operator_host(unsigned op, unsigned t, void* state, ITYPE dim,
                                                          void* stream, unsigned dev) {
    if (op == 0) return state_norm_squared_host(state, dim, stream, dev);
    return expectation_value_multi_qubit_Pauli_operator_partial_list_host(&t, &op, 1, state, dim, stream, dev);
}

qm_complex transition_amplitude_multi_qubit_Pauli_operator_XZ_mask_host(ITYPE bf, ITYPE pf, UINT rot, UINT pivot,
                                                                        void* bra, void* ket, ITYPE dim,
                                                                        void* stream, unsigned dev) {
    if (bf == 0) {
        set_error(QM_ERR_INVALID_ARGUMENT, "transition amplitude XZ mask: empty bit-flip mask");
        return qm_complex{0, 0};
    }
    return transition(make_term(bf, pf, rot, pivot), bra, ket, dim, stream, dev,
                      "transition_amplitude_multi_qubit_Pauli_operator_XZ_mask_host");
}
qm_complex transition_amplitude_multi_qubit_Pauli_operator_Z_mask_host(ITYPE pf, void* bra, void* ket, ITYPE dim,
                                                                       void* stream, unsigned dev) {
    return transition(make_term(0, pf, 0, 0), bra, ket, dim, stream, dev,
                      "transition_amplitude_multi_qubit_Pauli_operator_Z_mask_host");
}
qm_complex transition_amplitude_multi_qubit_Pauli_operator_partial_list_host(const UINT* tl, const UINT* pl, UINT n,
                                                                             void* bra, void* ket, ITYPE dim,
                                                                             void* stream, unsigned dev) {
    const char* what = "transition_amplitude_multi_qubit_Pauli_operator_partial_list_host";
    if (!state_ok(ket, dim, what)) return qm_complex{0, 0};
    Term t;
    if (!pauli_term_from_list(tl, pl, n, log2_dim(dim), &t, what)) return qm_complex{0, 0};
    return transition(t, bra, ket, dim, stream, dev, what);
}
qm_complex transition_amplitude_multi_qubit_Pauli_operator_whole_list_host(const UINT* pl, UINT n, void* bra,
                                                                           void* ket, ITYPE dim, void* stream,
                                                                           unsigned dev) {
    std::vector<u32> tl(n);
    for (UINT i = 0; i < n; ++i) tl[i] = i;
    return transition_amplitude_multi_qubit_Pauli_operator_partial_list_host(tl.data(), pl, n, bra, ket, dim, stream,
                                                                             dev);
}

qm_complex inner_product_host(const void* bra, const void* ket, ITYPE dim, void* stream, unsigned dev) {
    qm_complex z{0, 0};
    if (!state_ok(bra, dim, "inner_product_host") || !state_ok(ket, dim, "inner_product_host") || !use_device(dev))
        return z;
    RArgs r{};
    r.a = (const double2*)ket;
    r.b = (const double2*)bra;
    r.dim = dim;
    double res[2] = {0, 0};
    if (run_reduce<R_INNER>(r, dim, nullptr, stream_of(stream), res)) {
        z.re = res[0];
        z.im = res[1];
    }
    return z;
}

qm_complex qm_observable_expectation_host(const ITYPE* bfs, const ITYPE* pfs, const UINT* rots,
                                          const qm_complex* coefs, UINT nterms, void* state, ITYPE dim,
                                          void* stream, unsigned dev) {
    const char* what = "qm_observable_expectation_host";
    qm_complex z{0, 0};
    if (!state_ok(state, dim, what)) return z;
    if (nterms == 0) return z;
    if (!bfs || !pfs || !rots || !coefs) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null term arrays", what);
        return z;
    }
    if (!use_device(dev)) return z;
    const int n = log2_dim(dim);
    for (UINT k = 0; k < nterms; ++k)
        if (((bfs[k] | pfs[k]) >> n) != 0) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: term %u acts beyond %d qubits", what, k, n);
            return z;
        }
    hipStream_t st = stream_of(stream);
    Scratch* sc = scratch_for(st);
    if (!sc) return z;
    double total_re = 0, total_im = 0;
    // as many terms at a time as the upload ring takes
    const UINT chunk = 1u << 15;
    for (UINT off = 0; off < nterms; off += chunk) {
        const UINT cnt = std::min(chunk, nterms - off);
        const ObsPlan pl = plan_observable(bfs + off, pfs + off, rots + off, coefs + off, cnt, n);
        const ObsTerm* dt = nullptr;
        const ObsGroup* dg = nullptr;
        if (!obs_inline(pl) && !upload_plan(sc, pl, &dt, &dg)) return z;
        for (size_t g = 0; g < pl.groups.size(); g += pl.per_launch()) {
            if (!launch_observable(pl, g, std::min(pl.per_launch(), pl.groups.size() - g), state, dim, st,
                                   sc->partials, dt, dg, sc->host_result, what) ||
                !hip_ok(hipStreamSynchronize(st), what))
                return z;
            total_re += sc->host_result[0];
            total_im += sc->host_result[1];
        }
    }
    z.re = total_re;
    z.im = total_im;
    return z;
}

// ------------------------------------------------------------------ allocation-free observable
qm_complex qm_observable_expectation_noalloc_host(const ITYPE* bfs, const ITYPE* pfs, const UINT* rots,
                                                 const qm_complex* coefs, UINT nterms, void* state, ITYPE dim,
                                                 void* stream, unsigned dev) {
    const char* what = "qm_observable_expectation_noalloc_host";
    qm_complex z{0, 0};
    if (!state_ok(state, dim, what)) return z;
    if (nterms == 0) return z;
    if (!bfs || !pfs || !rots || !coefs) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null term arrays", what);
        return z;
    }
    if (nterms > kNoAllocMaxTerms) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: %u terms exceed the %u this entry point holds", what, nterms,
                  kNoAllocMaxTerms);
        return z;
    }
    const int n = log2_dim(dim);
    for (UINT k = 0; k < nterms; ++k)
        if (((bfs[k] | pfs[k]) >> n) != 0) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: term %u acts beyond %d qubits", what, k, n);
            return z;
        }
    const ObsPlan pl = plan_observable(bfs, pfs, rots, coefs, nterms, n);  // at most a group per term
    if (!use_device(dev)) return z;
    unsigned char* base = noalloc_scratch(dev, what);
    if (!base) return z;
    double* dout = (double*)(base + kNoAllocOutOff);
    hipStream_t st = stream_of(stream);
    ObsTerm* dt = nullptr;
    ObsGroup* dg = nullptr;
    if (!obs_inline(pl)) {
        dt = (ObsTerm*)(base + kNoAllocTermsOff);
        dg = (ObsGroup*)(base + kNoAllocGroupsOff);
        if (!hip_ok(hipMemcpyAsync(dt, pl.terms.data(), pl.terms.size() * sizeof(ObsTerm), hipMemcpyHostToDevice, st), what) ||
            !hip_ok(hipMemcpyAsync(dg, pl.groups.data(), pl.groups.size() * sizeof(ObsGroup), hipMemcpyHostToDevice, st),
                    what))
            return z;
    }
    double res[2] = {0, 0};
    if (!launch_observable(pl, 0, pl.groups.size(), state, dim, st, (double*)(base + kNoAllocPartialsOff), dt, dg, dout,
                           what) ||
        !hip_ok(hipMemcpyAsync(res, dout, sizeof(res), hipMemcpyDeviceToHost, st), what) ||
        !hip_ok(hipStreamSynchronize(st), what))
        return z;
    z.re = 0.0 + res[0];  // summed as in the allocating entry point
    z.im = 0.0 + res[1];
    return z;
}

// ------------------------------------------------------------------ state arithmetic
void normalize_host(double squared_norm, void* state, ITYPE dim, void* stream, unsigned dev) {
    if (!state_ok(state, dim, "normalize_host") || !use_device(dev)) return;
    hipStream_t st = stream_of(stream);
    const double f = std::sqrt(1.0 / squared_norm);  // src/csim/update_ops_named_state.cpp:23
    k_scale_r<<<grid_for(dim >> 1, 512), 512, 0, st>>>((double2*)state, dim, f);
    finish_update(st, "normalize_host");
}
void state_add_host(void* added, void* state, ITYPE dim, void* stream, unsigned dev) {
    if (!state_ok(state, dim, "state_add_host") || !state_ok(added, dim, "state_add_host") || !use_device(dev)) return;
    hipStream_t st = stream_of(stream);
    k_add<<<grid_for(dim, 256 * 4), 256, 0, st>>>((double2*)state, (const double2*)added, dim);
    finish_update(st, "state_add_host");
}
void qm_state_add_with_coef_host(qm_complex coef, const void* added, void* state, ITYPE dim, void* stream,
                                 unsigned dev) {
    if (!state_ok(state, dim, "qm_state_add_with_coef_host") || !state_ok(added, dim, "qm_state_add_with_coef_host") ||
        !use_device(dev))
        return;
    hipStream_t st = stream_of(stream);
    k_axpy<<<grid_for(dim, 256 * 4), 256, 0, st>>>((double2*)state, (const double2*)added, dim,
                                                    make_double2(coef.re, coef.im));
    finish_update(st, "qm_state_add_with_coef_host");
}
void state_multiply_host(qm_complex coef, void* state, ITYPE dim, void* stream, unsigned dev) {
    if (!state_ok(state, dim, "state_multiply_host") || !use_device(dev)) return;
    hipStream_t st = stream_of(stream);
    k_scale_c<<<grid_for(dim >> 1, 512), 512, 0, st>>>((double2*)state, dim, make_double2(coef.re, coef.im));
    finish_update(st, "state_multiply_host");
}

}  // extern "C"
