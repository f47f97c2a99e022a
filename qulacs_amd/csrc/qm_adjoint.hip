// Adjoint differentiation of <psi(theta)| H |psi(theta)> for circuits of fixed
// gates and parametric Pauli rotations, batched over parameter sets.
//
// Reference: ParametricQuantumCircuit::backprop / backprop_inner_product
// (src/vqcsim/parametric_circuit.cpp:205-335): run the circuit, set the
// "bistate" to 2 H|psi>, then walk the gates backwards applying each inverse to
// both states; at a parametric rotation R(theta) = exp(i theta P / 2) the
// gradient is Re <bistate| R(theta + pi) |state> / 2 = -Im <lambda|P|psi> with
// lambda = H|psi> (the reference's bistate is 2 lambda).  The reference spends
// a state copy, a gate and an inner product per parameter (about three passes)
// plus two more passes for the inverses.
//
// Here every gate becomes single-qubit operations, CZ gates and 4 x 4 matrices,
// and the tile engine (qm_tile.hpp) runs them stage by stage on tiles in LDS:
//   * a rotation about a Pauli string of several qubits is one RX between CZ gates
//     to its other qubits (CZ_{a,t} X_t CZ_{a,t} = X_t Z_a), after fixed
//     single-qubit changes of basis; CNOT is H CZ H;
//   * consecutive single-qubit gates on one qubit are one operation U = F_m ... F_1.
//     Its 2 x 2 matrix depends on the parameter set: k_adj_mats forms U and U^dagger
//     of every operation and set once per call;
//   * backward, the three numbers s_P = Im <lambda|P|psi>, P in {X, Y, Z} on the
//     operation's qubit after U, give the gradient of every rotation inside U: for
//     F_j = exp(i a P_j / 2) it is -sum_P g_P s_P with F_m..F_{j+1} P_j
//     (F_m..F_{j+1})^dagger = g_X X + g_Y Y + g_Z Z (k_adj_mats forms g).  A fused
//     RZ RY costs 12 multiply-adds per amplitude pair for its two gradients.
//
// Bound: FP64 issue and LDS round trips.  20 qubits, 12 layers of RY RZ and a CZ chain, 16
// parameter sets (256 MiB per state array): 42.3 ms with one kernel per 3-qubit register block
// straight from memory (160 passes at 3.0-3.6 TB/s), 11.3 ms with tiles in the order of the gate
// list (21 forward and 24 backward stages), 7.5 ms with Picker's 7 and 8 stages.
//
// Layout: `batch` states of 2^max(n, 4) complex128 each, contiguous (state b at
// b * dim); theta is batch x params (row-major).  Every reduction is a fixed-order
// sum of partial sums, so the results do not depend on scheduling, and a parameter
// set's result does not depend on the batch it is in.
#include "qm_tile.hpp"

namespace qm {
namespace {

constexpr int kAdjK = 3;             // block qubits of a pass: 8 amplitudes of psi and of lambda per thread
constexpr u32 kFwdLocal = 12;        // forward window: 64 KiB of psi
constexpr u32 kBwdLocal = 11;        // backward window: 32 KiB of psi and 32 KiB of lambda
constexpr u32 kFwdThreads = 1u << (kFwdLocal - kAdjK);
constexpr u32 kBwdThreads = 1u << (kBwdLocal - kAdjK);
constexpr u32 kStageGrads = 64;      // operations with gradients per backward stage (LDS sums)
constexpr u32 kChunkCols = 1536;     // columns of partial sums held at a time (at least a stage's, 3 * kStageGrads)
constexpr u64 kBwdMaxBlocks = 4096;  // work-groups per state of a backward stage (more tiles: several each)
constexpr u32 kHpsiThreads = 256;
constexpr u32 kHpsiMaxBlocks = 512;
// the neighbours of 1/sqrt(2), and what the upper one, which is nearer, has too much
constexpr double kRootHigh = 0.70710678118654757, kRootLow = 0.70710678118654746;
constexpr double kRootRest = -4.8336466567264567e-17;

// One factor of a single-qubit operation.
struct Factor {
    // 0: fixed matrix, 1 / 2 / 3: exp(i a P / 2) with P = X / Y / Z, 4: fixed matrix over sqrt(2)
    u32 kind;
    u32 fixed;   // kinds 0 and 4: offset into the fixed-matrix pool
    u32 param;   // rotation: parameter index
    u32 occ;     // rotation: occurrence number
    double coef; // rotation: a = coef * theta[param]
    __host__ __device__ bool rotation() const { return kind >= 1 && kind <= 3; }
};

struct AdjTerm {
    u64 pf;
    u32 rot, pad;
    double coef;
};
// terms [term0, term0 + nterm) share the bit-flip mask bf
struct AdjGroup {
    u64 bf;
    u32 term0, nterm;
};

__device__ __forceinline__ double2 ipow(double2 z, u32 k) {  // z * i^k
    switch (k & 3u) {
        case 0: return z;
        case 1: return make_double2(-z.y, z.x);
        case 2: return make_double2(-z.x, -z.y);
        default: return make_double2(z.y, -z.x);
    }
}

// hi + lo: a number of about 106 bits; lo is at most half a unit of hi's last place once
// `settle` has run.
struct Wide {
    double hi, lo;
};
__device__ __forceinline__ Wide settle(Wide a) {
#pragma clang fp contract(off)
    const double s = a.hi + a.lo;
    return Wide{s, a.lo - (s - a.hi)};
}
// acc + a b (b a plain number); contraction would turn the exact differences into something else
__device__ __forceinline__ Wide wide_mac(Wide acc, Wide a, double b) {
#pragma clang fp contract(off)
    const double p = a.hi * b, e = __builtin_fma(a.hi, b, -p);
    const double s = acc.hi + p, t = s - acc.hi;
    const double d = (acc.hi - (s - t)) + (p - t);
    return Wide{s, acc.lo + (d + __builtin_fma(a.lo, b, e))};
}
// u <- u m, 2 x 2 complex
__device__ __forceinline__ void wide_mul2(Wide (&re)[4], Wide (&im)[4], const double2 (&m)[4]) {
    Wide r[4], i[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int row = k & 2, col = k & 1;
        Wide x = wide_mac(Wide{0.0, 0.0}, re[row], m[col].x), y = wide_mac(Wide{0.0, 0.0}, re[row], m[col].y);
        x = wide_mac(x, im[row], -m[col].y);
        y = wide_mac(y, im[row], m[col].x);
        x = wide_mac(x, re[row + 1], m[2 + col].x);
        y = wide_mac(y, re[row + 1], m[2 + col].y);
        r[k] = settle(wide_mac(x, im[row + 1], -m[2 + col].y));
        i[k] = settle(wide_mac(y, im[row + 1], m[2 + col].x));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        re[k] = r[k];
        im[k] = i[k];
    }
}

// The matrices of every single-qubit operation for every parameter set: U into the
// forward pool, U^dagger into the backward pool, and per rotation occurrence the
// vector g (see the file comment).  blockIdx.y = set; one thread per operation.
// `copies` lists the pool entries that do not depend on the set (4 x 4 matrices).
//
// Products are formed in pairs of doubles and rounded once: an operation has the error of one
// gate, whatever it was made of.  The factors 1/sqrt(2) of the Hadamards that come with a CNOT or a
// Pauli string are left out and put in at the end, where pairs of them are exact; rounded, each
// would change the norm by up to 9e-17, always the same way, and the sweep back multiplies by the
// conjugate transposes, which doubles the change instead of undoing it.  6 qubits, 12 layers of RY RZ
// and a CNOT chain, error of the gradient against 80 bits: gate by gate 1.9e-15, products and
// Hadamards in double 5.7e-15, so 1.95e-15.
struct MatsArgs {
    const Factor* factors;
    const u32* first;      // factors [first[o], first[o + 1]) of operation o, in gate order
    const double2* fixed;  // fixed factors' matrices
    const u32* fwd_at;     // pool offsets of operation o's matrix
    const u32* bwd_at;
    const u32* copies;     // ncopy_f forward offsets, then ncopy_b backward offsets
    const double2* copy_val;
    const u32* low;        // operation o is a Hadamard that takes the lower neighbour of 1/sqrt(2)
    u32 nops, ncopy_f, ncopy_b, nparams, nocc;
    u32 fwd_stride, bwd_stride;
};
__global__ __launch_bounds__(64) void k_adj_mats(MatsArgs a, const double* __restrict__ theta, double2* __restrict__ fwd,
                                                 double2* __restrict__ bwd, double* __restrict__ gvec) {
    const u32 set = blockIdx.y, o = blockIdx.x * blockDim.x + threadIdx.x;
    double2* pf = fwd + (u64)set * a.fwd_stride;
    double2* pb = bwd + (u64)set * a.bwd_stride;
    if (o >= a.nops) {
        const u32 c = o - a.nops;
        if (c < a.ncopy_f) pf[a.copies[c]] = a.copy_val[c];
        else if (c < a.ncopy_f + a.ncopy_b) pb[a.copies[c]] = a.copy_val[c];
        return;
    }
    // sqrt(2)^roots u = F_m ... F_{j+1} while the factors are walked from the last to the first
    Wide ur[4] = {{1.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}, {1.0, 0.0}}, ui[4] = {};
    double half = 1.0;  // 2^-roots
    u32 roots = 0;
    for (u32 j = a.first[o + 1]; j-- > a.first[o];) {
        const Factor f = a.factors[j];
        // m = c I + i s P for a rotation about P = X, Y or Z (px, py, pz); selected without
        // branches
        const double px = f.kind == 1 ? 1.0 : 0.0, py = f.kind == 2 ? 1.0 : 0.0, pz = f.kind == 3 ? 1.0 : 0.0;
        double2 m[4];
        if (!f.rotation()) {
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = a.fixed[f.fixed + i];
            half *= f.kind == 4 ? 0.5 : 1.0;
            roots += f.kind == 4 ? 1u : 0u;
        } else {
            double2 u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = make_double2(ur[i].hi, ui[i].hi);
            // u P u^dagger = [[g_Z, g_X - i g_Y], [g_X + i g_Y, -g_Z]], from its entries (0, 0) and (1, 0)
            const double2 c0 = cconj(u[0]), c1 = cconj(u[1]);
            const double2 z20 = cmul(u[2], c0), z21 = cmul(u[2], c1), z30 = cmul(u[3], c0), z31 = cmul(u[3], c1);
            const double2 z01 = cmul(u[0], c1);
            const double n0 = u[0].x * u[0].x + u[0].y * u[0].y, n1 = u[1].x * u[1].x + u[1].y * u[1].y;
            double* g = gvec + ((u64)set * a.nocc + f.occ) * 3;
            g[0] = half * (px * (z30.x + z21.x) - py * (z30.y - z21.y) + pz * (z20.x - z31.x));
            g[1] = half * (px * (z30.y + z21.y) + py * (z30.x - z21.x) + pz * (z20.y - z31.y));
            g[2] = half * (2.0 * (px * z01.x + py * z01.y) + pz * (n0 - n1));
            const double ang = 0.5 * (f.coef * theta[(u64)set * a.nparams + f.param]);
            const double c = cos(ang), s = sin(ang);
            m[0] = make_double2(c, s * pz);
            m[1] = make_double2(s * py, s * px);
            m[2] = make_double2(-(s * py), s * px);
            m[3] = make_double2(c, -(s * pz));
        }
        wide_mul2(ur, ui, m);
    }
    // times 2^-(roots / 2), and 1/sqrt(2) for an odd one
    const double pairs = ldexp(1.0, -(int)(roots / 2));
    const bool odd = roots & 1u, low = a.low[o];
    const double rh = odd ? (low ? kRootLow : kRootHigh) : 1.0, rl = odd && !low ? kRootRest : 0.0;
    double2 u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const Wide x = wide_mac(wide_mac(Wide{0.0, 0.0}, ur[i], rl), ur[i], rh);
        const Wide y = wide_mac(wide_mac(Wide{0.0, 0.0}, ui[i], rl), ui[i], rh);
        u[i] = make_double2(pairs * (x.hi + x.lo), pairs * (y.hi + y.lo));
    }
    double2* uf = pf + a.fwd_at[o];
    double2* ub = pb + a.bwd_at[o];
    uf[0] = u[0]; uf[1] = u[1]; uf[2] = u[2]; uf[3] = u[3];
    ub[0] = cconj(u[0]); ub[1] = cconj(u[2]); ub[2] = cconj(u[1]); ub[3] = cconj(u[3]);
}

// One forward stage: a work-group per tile (blockIdx.x) and set (blockIdx.y).  Two
// groups of 64 KiB share a CU, so one's loads and stores overlap the other's passes.
// `first`: the tile is a part of |0...0>, nothing is read.
__global__ __launch_bounds__(kFwdThreads, 4) void k_adj_fwd(double2* __restrict__ psi, u32 n, u32 lq, u32 first,
                                                            DStage sg, const DPass* __restrict__ passes,
                                                            const DSub* __restrict__ subs,
                                                            const double2* __restrict__ pool, u32 stride) {
    extern __shared__ double2 st[];
    __shared__ u64 hi_tab[1u << (kFwdLocal - kLowFixed)];
    const u32 L = 1u << lq, T = blockDim.x;
    double2* s = psi + ((u64)blockIdx.y << n);
    build_hi_tab(hi_tab, lq, sg);
    const u64 tb = tile_base(blockIdx.x, n - lq, sg);
    __syncthreads();
    if (sg.npass) warm_program(passes[sg.pass0], subs, pool + (u64)blockIdx.y * stride);
    if (first) {
        for (u32 i = threadIdx.x; i < L; i += T)
            st[slot_of(i)] = make_double2(i == 0 && blockIdx.x == 0 ? 1.0 : 0.0, 0.0);
    } else if (L == 8 * kFwdThreads) {
#pragma unroll
        for (u32 k = 0; k < 8; ++k) {
            const u32 i = threadIdx.x + k * kFwdThreads;
            st[slot_of(i)] = s[tile_index(tb, hi_tab, i)];
        }
    } else {
        for (u32 i = threadIdx.x; i < L; i += T) st[slot_of(i)] = s[tile_index(tb, hi_tab, i)];
    }
    __syncthreads();
    run_passes<kAdjK, kFwdThreads, 1, false>(st, lq, passes, sg.pass0, sg.npass, subs,
                                             pool + (u64)blockIdx.y * stride, blockIdx.x);
    for (u32 i = threadIdx.x; i < L; i += T) s[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
}

// Wave sums of a, b, c: afterwards every lane of row r (16 lanes) holds the sum of a, b, c
// for r = 0, 1, 2.  Two swap levels put different values into the rows, so four row levels serve
// all three: 21 vector instructions instead of 54 for three separate sums.
__device__ __forceinline__ double swap_add32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((u32)__double2loint(a), (u32)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((u32)__double2hiint(a), (u32)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((u32)__double2loint(a), (u32)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((u32)__double2hiint(a), (u32)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum3(double a, double b, double c) {
    double v = swap_add16(swap_add32(a, c), swap_add32(b, 0.0));
    v = dpp_add<0x128>(v);  // row_ror:8
    v = dpp_add<0x124>(v);  // row_ror:4
    v = dpp_add<0x122>(v);  // row_ror:2
    return dpp_add<0x121>(v);
}

// One bit of a backward LAYER: the three sums of its operation (if it has gradients), then
// U^dagger on psi (v) and lambda (l).  out: this wave's sums of the operation in LDS.
template <int P>
__device__ __forceinline__ void bwd_bit(double2 (&v)[1 << kAdjK], double2 (&l)[1 << kAdjK], const double2* mp,
                                        bool grad, bool add, double* out) {
    constexpr int NP = 1 << (kAdjK - 1);
    const double2 m0 = mp[0], m1 = mp[1], m2 = mp[2], m3 = mp[3];
    auto pair_j = [](int q) { return ((q >> P) << (P + 1)) | (q & ((1 << P) - 1)); };
    if (grad) {
        double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const double2 a = v[pair_j(q)], b = v[pair_j(q) | (1 << P)];
            const double2 c = l[pair_j(q)], d = l[pair_j(q) | (1 << P)];
            sx = fma(c.x, b.y, sx); sy = fma(-c.x, b.x, sy); sz = fma(c.x, a.y, sz);
            sx = fma(-c.y, b.x, sx); sy = fma(-c.y, b.y, sy); sz = fma(-c.y, a.x, sz);
            sx = fma(d.x, a.y, sx); sy = fma(d.x, a.x, sy); sz = fma(-d.x, b.y, sz);
            sx = fma(-d.y, a.x, sx); sy = fma(d.y, a.y, sy); sz = fma(d.y, b.x, sz);
        }
        const double r = wave_sum3(sx, sy, sz);
        const u32 lane = threadIdx.x & 63u;
        if ((lane & 15u) == 0 && lane < 48) {
            if (add) out[lane >> 4] += r;
            else out[lane >> 4] = r;
        }
    }
#pragma unroll
    for (int q = 0; q < NP; ++q)
        pair_update2(v[pair_j(q)], v[pair_j(q) | (1 << P)], l[pair_j(q)], l[pair_j(q) | (1 << P)], m0, m1, m2, m3);
}

// One backward stage: as k_adj_fwd on the tiles of psi and lambda, the operations reversed and
// inverted.  A thread holds one register block of each state; the tile has at most T blocks
// (threads beyond them hold zeros, so that the wave sums see every lane).  Work-group x takes
// tiles x, x + gridDim.x, ... and writes its sums of the stage's operations to
// partials[set][x][col0 ..].
__global__ __launch_bounds__(kBwdThreads, 2) void k_adj_bwd(double2* __restrict__ psi, double2* __restrict__ lam, u32 n,
                                                            u32 lq, u64 ntiles, DStage sg, u32 grad0, u32 ngrad, u32 col0,
                                                            const DPass* __restrict__ passes,
                                                            const DSub* __restrict__ subs,
                                                            const double2* __restrict__ pools, u32 stride,
                                                            double* __restrict__ partials, u32 ncols) {
    extern __shared__ double2 st[];
    __shared__ u64 hi_tab[1u << (kBwdLocal - kLowFixed)];
    __shared__ double acc[kBwdThreads / 64][kStageGrads][3];
    constexpr int D = 1 << kAdjK;
    const u32 L = 1u << lq, T = blockDim.x, tid = threadIdx.x, wave = tid >> 6;
    const u32 ngroups = L >> kAdjK;
    const double2* __restrict__ pool = pools + (u64)blockIdx.y * stride;
    double2* P = psi + ((u64)blockIdx.y << n);
    double2* Q = lam + ((u64)blockIdx.y << n);
    double2* st2 = st + L;
    build_hi_tab(hi_tab, lq, sg);
    __syncthreads();
    for (u64 t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const bool add = t != blockIdx.x;  // a later tile of this work-group
        const u64 tb = tile_base(t, n - lq, sg);
        if (L == 8 * kBwdThreads) {
#pragma unroll
            for (u32 k = 0; k < 8; ++k) {
                const u32 i = tid + k * kBwdThreads;
                const u64 at = tile_index(tb, hi_tab, i);
                st[slot_of(i)] = P[at];
                st2[slot_of(i)] = Q[at];
            }
        } else {
            for (u32 i = tid; i < L; i += T) {
                const u64 at = tile_index(tb, hi_tab, i);
                st[slot_of(i)] = P[at];
                st2[slot_of(i)] = Q[at];
            }
        }
        __syncthreads();
        for (u32 p = 0; p < sg.npass; ++p) {
            const DPass ps = passes[sg.pass0 + p];
            if (ps.warm) warm_program(ps, subs, pool);
            const bool mine = tid < ngroups;
            u32 base = mine ? tid : 0, slot[D];
#pragma unroll
            for (int i = 0; i < kAdjK; ++i) {
                const u32 q = ps.pos[i];
                base = (base & ((1u << q) - 1)) | ((base >> q) << (q + 1));
            }
            slot[0] = slot_of(base);
#pragma unroll
            for (int j = 1; j < D; ++j) {
                slot[j] = slot[j & (j - 1)] ^ ps.sbit[__builtin_ctz(j)];
                asm volatile("" : "+v"(slot[j]));
            }
            double2 v[D], l[D];
#pragma unroll
            for (int j = 0; j < D; ++j) {
                v[j] = st[slot[j]];
                l[j] = st2[slot[j]];
            }
            if (!mine) {
#pragma unroll
                for (int j = 0; j < D; ++j) v[j] = l[j] = make_double2(0.0, 0.0);
            }
            u32 k = 0;
            while (k < ps.nsub) {
                DSub sub = subs[ps.sub0 + k];
                while ((sub.type & 15u) == SUB_LAYER) {
                    const u32 d1 = (sub.type >> 8) & 15u;
                    if ((sub.type >> 12) | sub.nx) {
                        const u32 sgn = layer_signs<kAdjK>(sub, base, t);
                        flip_signs<kAdjK>(v, sgn);
                        flip_signs<kAdjK>(l, sgn);
                    }
                    const double2* mp = pool + sub.data;
                    double* out = acc[wave][sub.grad0 - grad0];
                    if (d1 & 1u) {
                        bwd_bit<0>(v, l, mp, sub.gmask & 1u, add, out);
                        mp += 4;
                        out += 3 * (sub.gmask & 1u);
                    }
                    if (d1 & 2u) {
                        bwd_bit<1>(v, l, mp, sub.gmask & 2u, add, out);
                        mp += 4;
                        out += 3 * ((sub.gmask >> 1) & 1u);
                    }
                    if (d1 & 4u) bwd_bit<2>(v, l, mp, sub.gmask & 4u, add, out);
                    if (++k == ps.nsub) break;
                    sub = subs[ps.sub0 + k];
                }
                if (k == ps.nsub) break;
                // D2: the 4 x 4 matrix on both states
                const double2* mp = pool + sub.data;
                apply_d2<kAdjK>(v, byte_at(sub.a, 0), byte_at(sub.a, 1), mp);
                apply_d2<kAdjK>(l, byte_at(sub.a, 0), byte_at(sub.a, 1), mp);
                ++k;
            }
            if (mine) {
#pragma unroll
                for (int j = 0; j < D; ++j) {
                    st[slot[j]] = v[j];
                    st2[slot[j]] = l[j];
                }
            }
            __syncthreads();
        }
        for (u32 i = tid; i < L; i += T) {
            const u64 at = tile_index(tb, hi_tab, i);
            P[at] = st[slot_of(i)];
            Q[at] = st2[slot_of(i)];
        }
        __syncthreads();  // the tile has been read out of LDS
    }
    double* dst = partials + ((u64)blockIdx.y * gridDim.x + blockIdx.x) * ncols + col0;
    for (u32 i = tid; i < 3 * ngrad; i += T) {
        double s = 0.0;
        for (u32 w = 0; w < T / 64; ++w) s += acc[w][i / 3][i % 3];
        dst[i] = s;
    }
}

// lambda = sum_k c_k P_k psi and the block's share of Re <psi|lambda>.  Terms with one
// bit-flip mask read their partner amplitude once.
__global__ __launch_bounds__(kHpsiThreads) void k_adj_hpsi(const double2* __restrict__ psi, double2* __restrict__ lam,
                                                           u64 dim, const AdjGroup* __restrict__ groups, u32 ngroup,
                                                           const AdjTerm* __restrict__ terms,
                                                           double* __restrict__ epart) {
    __shared__ double red[32];
    const u64 off = (u64)blockIdx.y * dim;
    const double2* P = psi + off;
    double acc = 0.0;
    for (u64 x = (u64)blockIdx.x * blockDim.x + threadIdx.x; x < dim; x += (u64)gridDim.x * blockDim.x) {
        double2 s = make_double2(0.0, 0.0);
        for (u32 g = 0; g < ngroup; ++g) {
            const AdjGroup gr = groups[g];
            const u64 y = x ^ gr.bf;
            const double2 v = P[y];
            double2 c = make_double2(0.0, 0.0);  // sum_k c_k i^rot (-1)^popcount(y & pf)
            for (u32 k = 0; k < gr.nterm; ++k) {
                const AdjTerm tm = terms[gr.term0 + k];
                const double sg = (__popcll(y & tm.pf) & 1) ? -tm.coef : tm.coef;
                const double2 f = ipow(make_double2(1.0, 0.0), tm.rot);
                c.x = fma(sg, f.x, c.x);
                c.y = fma(sg, f.y, c.y);
            }
            s = cmac(s, c, v);
        }
        lam[off + x] = s;
        const double2 p = P[x];
        acc += p.x * s.x + p.y * s.y;
    }
    acc = block_sum(acc, red);
    if (threadIdx.x == 0) epart[(u64)blockIdx.y * gridDim.x + blockIdx.x] = acc;
}

// Columns of partials[set][block][ncols] summed over the blocks into sums[set][total], from
// sums + col0 on: 16 columns per work-group, 16 threads per column, each over every 16th block,
// then in order.
__global__ __launch_bounds__(256) void k_adj_columns(const double* __restrict__ partials, u32 nblk, u32 ncols,
                                                     double* __restrict__ sums, u32 total, u32 col0) {
    __shared__ double red[16][17];
    const u32 c = threadIdx.x & 15u, part = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
    const double* src = partials + (u64)blockIdx.y * nblk * ncols;
    double s = 0.0;
    if (col < ncols)
        for (u32 b = part; b < nblk; b += 16) s += src[(u64)b * ncols + col];
    red[part][c] = s;
    __syncthreads();
    if (part == 0 && col < ncols) {
        double r = 0.0;
        for (u32 k = 0; k < 16; ++k) r += red[k][c];
        sums[(u64)blockIdx.y * total + col0 + col] = r;
    }
}

// grad[set][p] = -sum over the occurrences of p (in order) of coef * (g . s); the first
// thread of a set's first block adds up its energy.
__global__ __launch_bounds__(64) void k_adj_grad(const double* __restrict__ sums, u32 ncols,
                                                 const double* __restrict__ gvec, u32 nocc,
                                                 const u32* __restrict__ first, const u32* __restrict__ occs,
                                                 const u32* __restrict__ occ_col, const double* __restrict__ occ_coef,
                                                 u32 nparams, double* __restrict__ grad,
                                                 const double* __restrict__ epart, u32 neblk,
                                                 double* __restrict__ energy) {
    const u32 p = blockIdx.x * blockDim.x + threadIdx.x, set = blockIdx.y;
    if (blockIdx.x == 0) {  // the set's energy
        double e = 0.0;
        for (u32 k = threadIdx.x; k < neblk; k += 64) e += epart[(u64)set * neblk + k];
        e = wave_sum(e);
        if (threadIdx.x == 0) energy[set] = e;
    }
    if (p >= nparams) return;
    double r = 0.0;
    for (u32 k = first[p]; k < first[p + 1]; ++k) {
        const u32 o = occs[k];
        const double* g = gvec + ((u64)set * nocc + o) * 3;
        const double* s = sums + (u64)set * ncols + occ_col[o];
        r -= occ_coef[o] * (g[0] * s[0] + g[1] * s[1] + g[2] * s[2]);
    }
    grad[(u64)set * nparams + p] = r;
}

// ------------------------------------------------------------------ host side
// A single-qubit operation while the circuit is read: its factors in gate order.
struct Op1 {
    std::vector<Factor> factors;
    bool grad = false;
    bool given = false;  // has a rotation or a matrix of the caller's
    u32 roots = 0;       // factors of kind 4
};

bool unitary2(const cd* m) {
    const cd a = std::conj(m[0]) * m[0] + std::conj(m[2]) * m[2], b = std::conj(m[1]) * m[1] + std::conj(m[3]) * m[3];
    const cd c = std::conj(m[0]) * m[1] + std::conj(m[2]) * m[3];
    return std::abs(a - 1.0) < 1e-12 && std::abs(b - 1.0) < 1e-12 && std::abs(c) < 1e-12;
}

// The circuit as single-qubit operations, CZ gates and 4 x 4 matrices.
struct Builder {
    u32 ne = 0;
    std::vector<HOp> ops;
    std::vector<Op1> op1;
    std::vector<double2> fixed;
    std::vector<long> last;  // per qubit: index in ops of its last operation, if single-qubit and open
    std::vector<Factor> occ; // rotation occurrences

    explicit Builder(u32 n) : ne(n), last(n, -1) {}
    Op1& open(u32 q) {
        if (last[q] < 0) {
            HOp h;
            h.type = 0;
            h.q = {q};
            h.m.assign(4, 0.0);
            h.id = (long)op1.size();
            last[q] = (long)ops.size();
            ops.push_back(std::move(h));
            op1.emplace_back();
        }
        return op1[ops[last[q]].id];
    }
    void put1(u32 q, const cd* m) {
        // a matrix that is not unitary keeps an operation of its own: the gradient of a
        // rotation before it needs the state between the two
        const bool closed = !unitary2(m);
        if (closed) last[q] = -1;
        Factor f{};
        f.fixed = (u32)fixed.size();
        for (int i = 0; i < 4; ++i) fixed.push_back(make_double2(m[i].real(), m[i].imag()));
        Op1& o = open(q);
        o.factors.push_back(f);
        o.given = true;
        if (closed) last[q] = -1;
    }
    void cz(u32 a, u32 b) {
        HOp h;
        h.type = 2;
        h.q = {a, b};
        ops.push_back(std::move(h));
        last[a] = last[b] = -1;
    }
    void put2(u32 a, u32 b, const cd* m) {
        HOp h;
        h.type = 0;
        h.q = {a, b};
        h.m.assign(m, m + 16);
        ops.push_back(std::move(h));
        last[a] = last[b] = -1;
    }
    // A matrix of units (1, -1, i, -i and 0), over sqrt(2) if `root`.
    void put_units(u32 q, const cd (&m)[4], bool root) {
        Op1& o = open(q);
        Factor f{};
        f.kind = root ? 4 : 0;
        f.fixed = (u32)fixed.size();
        for (const cd& z : m) fixed.push_back(make_double2(z.real(), z.imag()));
        o.factors.push_back(f);
        o.roots += root;
    }
    void h(u32 q) { put_units(q, {1.0, 1.0, 1.0, -1.0}, true); }
    void rot1(u32 q, u32 pauli, u32 param, double coef) {
        Op1& o = open(q);
        Factor f{};
        f.kind = pauli;
        f.param = param;
        f.coef = coef;
        f.occ = (u32)occ.size();
        occ.push_back(f);
        o.factors.push_back(f);
        o.grad = o.given = true;
        ops[last[q]].grad = true;
    }
    // exp(i a P / 2), P a Pauli string on k >= 2 qubits
    void rotation(u32 k, const u32* q, const u32* pauli, u32 param, double coef) {
        u32 t = 0;  // the qubit that is rotated: one with an X if there is one, else a Z
        for (u32 j = 0; j < k; ++j)
            if (pauli[j] == 1 || (pauli[t] == 2 && pauli[j] == 3)) t = j;
        // basis changes to Z (other qubits) and X (qubit t) and back
        const cd i1(0, 1);
        auto change = [&](u32 j, bool back) {
            if (j == t) {
                if (pauli[j] == 3) h(q[j]);
                if (pauli[j] == 2) put_units(q[j], {1.0, 0.0, 0.0, back ? i1 : -i1}, false);  // diag(1, -i) Y diag(1, i) = X
            } else if (pauli[j] == 1) {
                h(q[j]);
            } else if (pauli[j] == 2) {
                // V = (1/sqrt2) [[1, -i], [1, i]]: V Y V^dagger = Z
                if (back) put_units(q[j], {1.0, 1.0, i1, -i1}, true);
                else put_units(q[j], {1.0, -i1, 1.0, i1}, true);
            }
        };
        for (u32 j = 0; j < k; ++j) change(j, false);
        for (u32 j = 0; j < k; ++j)
            if (j != t) cz(q[j], q[t]);
        rot1(q[t], 1, param, coef);
        for (u32 j = 0; j < k; ++j)
            if (j != t) cz(q[j], q[t]);
        for (u32 j = 0; j < k; ++j) change(j, true);
    }
};

template <class T>
bool put_dev(T** dst, const std::vector<T>& src, const char* what) {
    *dst = nullptr;
    if (src.empty()) return true;
    return hip_ok(hipMalloc((void**)dst, src.size() * sizeof(T)), what) &&
           hip_ok(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice), what);
}

}  // namespace
}  // namespace qm

using namespace qm;

struct qm_adjoint {
    u32 n = 0, ne = 0, nparams = 0, lqf = 0, lqb = 0;
    u64 ngates = 0;
    Flat fwd, bwd;
    std::vector<u32> stage_grad0;  // backward stage -> position in bwd.grads of its first operation
    // runs of backward stages whose partial sums share the workspace's columns: the first stage
    // of each, and the widest one's columns
    std::vector<u32> chunk0;
    u32 chunk_cols = 0;
    // host tables, uploaded on first use
    std::vector<Factor> factors;
    std::vector<u32> first, fwd_at, bwd_at, copies, low, par_first, par_occs, occ_col;
    std::vector<double2> fixed, copy_val;
    std::vector<double> occ_coef;
    u32 ncopy_f = 0, ncopy_b = 0;
    int device = -1;
    Factor* d_factors = nullptr;
    u32 *d_first = nullptr, *d_fwd_at = nullptr, *d_bwd_at = nullptr, *d_copies = nullptr, *d_low = nullptr, *d_par_first = nullptr,
        *d_par_occs = nullptr, *d_occ_col = nullptr;
    double2 *d_fixed = nullptr, *d_copy_val = nullptr;
    double* d_occ_coef = nullptr;
    DPass *d_fpass = nullptr, *d_bpass = nullptr;
    DSub *d_fsub = nullptr, *d_bsub = nullptr;

    u32 nops() const { return (u32)first.size() - 1; }
    u32 nocc() const { return (u32)occ_coef.size(); }
    u32 ncols() const { return 3 * (u32)bwd.grads.size(); }
    u64 tiles_b() const { return 1ULL << (ne - lqb); }
    u32 blocks_b() const { return (u32)std::min<u64>(tiles_b(), kBwdMaxBlocks); }
    u32 blocks_h() const {
        return (u32)std::min<u64>(std::max<u64>((1ULL << ne) / (4 * kHpsiThreads), 1), kHpsiMaxBlocks);
    }
    // workspace parts, in order; each a multiple of 16 bytes
    u64 state_bytes(u64 batch) const { return batch * (16ULL << ne); }
    u64 fpool_bytes(u64 batch) const { return batch * fwd.pool.size() * 16; }
    u64 bpool_bytes(u64 batch) const { return batch * bwd.pool.size() * 16; }
    u64 part_bytes(u64 batch) const { return (batch * blocks_b() * chunk_cols * 8 + 15) & ~15ULL; }
    u64 sums_bytes(u64 batch) const { return (batch * ncols() * 8 + 15) & ~15ULL; }
    u64 gvec_bytes(u64 batch) const { return (batch * nocc() * 24 + 15) & ~15ULL; }
    u64 epart_bytes(u64 batch) const { return (batch * blocks_h() * 8 + 15) & ~15ULL; }

    void release() {
        if (device >= 0) {
            (void)hipSetDevice(device);
            void* ptrs[] = {d_factors, d_first, d_fwd_at, d_bwd_at, d_copies, d_low, d_par_first, d_par_occs, d_occ_col,
                            d_fixed, d_copy_val, d_occ_coef, d_fpass, d_bpass, d_fsub, d_bsub};
            for (void* p : ptrs)
                if (p) (void)hipFree(p);
        }
        d_factors = nullptr; d_first = nullptr; d_fwd_at = nullptr; d_bwd_at = nullptr; d_copies = nullptr; d_low = nullptr;
        d_par_first = nullptr; d_par_occs = nullptr; d_occ_col = nullptr; d_fixed = nullptr; d_copy_val = nullptr;
        d_occ_coef = nullptr; d_fpass = nullptr; d_bpass = nullptr; d_fsub = nullptr; d_bsub = nullptr;
        device = -1;
    }
    bool prepare(unsigned dev, const char* what) {
        if (device == (int)dev) return true;
        release();
        device = (int)dev;  // release() frees what the uploads below allocate
        const bool ok = put_dev(&d_factors, factors, what) && put_dev(&d_first, first, what) &&
                        put_dev(&d_fwd_at, fwd_at, what) && put_dev(&d_bwd_at, bwd_at, what) &&
                        put_dev(&d_copies, copies, what) && put_dev(&d_low, low, what) && put_dev(&d_par_first, par_first, what) &&
                        put_dev(&d_par_occs, par_occs, what) && put_dev(&d_occ_col, occ_col, what) &&
                        put_dev(&d_fixed, fixed, what) && put_dev(&d_copy_val, copy_val, what) &&
                        put_dev(&d_occ_coef, occ_coef, what) && put_dev(&d_fpass, fwd.passes, what) &&
                        put_dev(&d_bpass, bwd.passes, what) && put_dev(&d_fsub, fwd.subs, what) &&
                        put_dev(&d_bsub, bwd.subs, what) &&
                        hip_ok(hipFuncSetAttribute((const void*)k_adj_fwd, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)(sizeof(double2) << kFwdLocal)), what) &&
                        hip_ok(hipFuncSetAttribute((const void*)k_adj_bwd, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)(2 * sizeof(double2) << kBwdLocal)), what);
        if (!ok) release();
        return ok;
    }
    void build(const Builder& b);
};

// Schedules the operations forward and, reversed and inverted, backward, and lays out the tables.
void qm_adjoint::build(const Builder& b) {
    lqf = std::min(ne, kFwdLocal);
    lqb = std::min(ne, kBwdLocal);
    HCirc hc;
    hc.n = hc.ne = ne;
    hc.ops = b.ops;
    schedule_circuit(fwd, hc, kAdjK, kFwdLocal);
    std::reverse(hc.ops.begin(), hc.ops.end());
    for (HOp& o : hc.ops)
        if (o.type == 0 && o.q.size() == 2) {  // 4 x 4: conjugate transpose
            const std::vector<cx> m = o.m;
            for (int r = 0; r < 4; ++r)
                for (int c = 0; c < 4; ++c) o.m[r * 4 + c] = std::conj(m[c * 4 + r]);
        }
    schedule_circuit(bwd, hc, kAdjK, kBwdLocal, kStageGrads);
    // first gradient of each backward stage: stages hold whole passes, in order
    stage_grad0.clear();
    u32 g = 0;
    for (const DStage& sg : bwd.stages) {
        stage_grad0.push_back(g);
        for (u32 p = 0; p < sg.npass; ++p) {
            const DPass& ps = bwd.passes[sg.pass0 + p];
            for (u32 k = 0; k < ps.nsub; ++k) g += (u32)__builtin_popcount(bwd.subs[ps.sub0 + k].gmask);
        }
    }
    stage_grad0.push_back(g);
    // Partial sums are blocks x columns: held for the whole sweep they would grow with the
    // circuit (40000 parameters at 20 qubits: 240 MiB beside 32 of states), so they are added up
    // when kChunkCols are full.  A launch of some microseconds per chunk; most circuits have one.
    chunk0.assign(1, 0);
    chunk_cols = 0;
    for (u32 s = 0; s < bwd.stages.size(); ++s) {
        if (3 * (stage_grad0[s + 1] - stage_grad0[chunk0.back()]) > kChunkCols) chunk0.push_back(s);
        chunk_cols = std::max(chunk_cols, 3 * (stage_grad0[s + 1] - stage_grad0[chunk0.back()]));
    }
    chunk0.push_back((u32)bwd.stages.size());
    factors.clear();
    first.assign(1, 0);
    for (const Op1& o : b.op1) {
        factors.insert(factors.end(), o.factors.begin(), o.factors.end());
        first.push_back((u32)factors.size());
    }
    // Hadamards on their own have the rounded 1/sqrt(2) as it is: each takes the neighbour that
    // keeps the product of all of them so far nearest to a unitary.
    low.assign(b.op1.size(), 0);
    double scale = 0.0;  // log of that product, relative to a unitary
    const double up = -kRootRest / kRootHigh, down = up - (kRootHigh - kRootLow) / kRootHigh;
    for (size_t o = 0; o < b.op1.size(); ++o) {
        if (b.op1[o].given || !(b.op1[o].roots & 1u)) continue;
        low[o] = std::abs(scale + down) < std::abs(scale + up);
        scale += low[o] ? down : up;
    }
    fixed = b.fixed;
    auto place = [&](const Flat& f, std::vector<u32>& at, u32& ncopy) {
        at.assign(b.op1.size(), 0);
        std::vector<bool> set(f.pool.size(), false);
        for (const auto& m : f.mats) {
            at[m.first] = m.second;
            for (u32 i = 0; i < 4; ++i) set[m.second + i] = true;
        }
        ncopy = 0;
        for (u32 i = 0; i < f.pool.size(); ++i)
            if (!set[i]) {
                copies.push_back(i);
                copy_val.push_back(f.pool[i]);
                ++ncopy;
            }
    };
    place(fwd, fwd_at, ncopy_f);
    place(bwd, bwd_at, ncopy_b);
    // column of each occurrence's operation, occurrences by parameter
    std::vector<u32> col(b.op1.size(), 0);
    for (size_t i = 0; i < bwd.grads.size(); ++i) col[bwd.grads[i]] = 3 * (u32)i;
    occ_col.assign(b.occ.size(), 0);
    occ_coef.assign(b.occ.size(), 0.0);
    for (size_t o = 0; o < b.op1.size(); ++o)
        for (const Factor& f : b.op1[o].factors)
            if (f.rotation()) {
                occ_col[f.occ] = col[o];
                occ_coef[f.occ] = f.coef;
            }
    par_first.assign((size_t)nparams + 1, 0);
    for (const Factor& f : b.occ) ++par_first[f.param + 1];
    for (u32 p = 0; p < nparams; ++p) par_first[p + 1] += par_first[p];
    par_occs.assign(b.occ.size(), 0);
    std::vector<u32> next(par_first.begin(), par_first.end() - 1);
    for (const Factor& f : b.occ) par_occs[next[f.param]++] = f.occ;  // occurrences in order
}

extern "C" {

qm_adjoint* qm_adjoint_create(UINT n, const qm_adjoint_gate* gates, UINT gate_count, UINT nparams) {
    const char* what = "qm_adjoint_create";
    if (n < 1 || n > 34 || (gate_count && !gates)) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: qubit count %u outside 1..34 or null gates", what, n);
        return nullptr;
    }
    const u32 ne = std::max<u32>(n, kMinQubits);
    Builder b(ne);
    for (UINT i = 0; i < gate_count; ++i) {
        const qm_adjoint_gate& in = gates[i];
        const u32 k = in.qubit_count;
        u64 mask = 0;
        bool ok = k >= 1 && k <= 4;
        for (u32 j = 0; ok && j < k; ++j) {
            ok = in.qubits[j] < n && !((mask >> in.qubits[j]) & 1);
            mask |= 1ULL << in.qubits[j];
        }
        if (ok && in.kind == QM_ADJ_ROT) {
            for (u32 j = 0; ok && j < k; ++j) ok = in.paulis[j] >= 1 && in.paulis[j] <= 3;
            ok = ok && in.param < nparams;
            if (ok && k == 1) b.rot1(in.qubits[0], in.paulis[0], in.param, in.coef);
            else if (ok) b.rotation(k, in.qubits, in.paulis, in.param, in.coef);
        } else if (ok) {
            const bool two = in.kind == QM_BATCH_CZ || in.kind == QM_BATCH_CNOT;
            ok = (in.kind <= QM_BATCH_CNOT) && (two ? k == 2 : k <= 2) && (two || in.matrix);
            if (ok && in.kind == QM_BATCH_CZ) {
                b.cz(in.qubits[0], in.qubits[1]);
            } else if (ok && in.kind == QM_BATCH_CNOT) {
                b.h(in.qubits[1]);
                b.cz(in.qubits[0], in.qubits[1]);
                b.h(in.qubits[1]);
            } else if (ok) {
                const u32 d = 1u << k;
                std::vector<cd> m((size_t)d * d, 0.0);
                for (u32 r = 0; r < d; ++r)
                    for (u32 c = 0; c < d; ++c) {
                        if (in.kind == QM_BATCH_DENSE) m[r * d + c] = cd(in.matrix[r * d + c].re, in.matrix[r * d + c].im);
                        else if (r == c) m[r * d + c] = cd(in.matrix[r].re, in.matrix[r].im);
                    }
                if (k == 1) b.put1(in.qubits[0], m.data());
                else b.put2(in.qubits[0], in.qubits[1], m.data());
            }
        }
        if (!ok) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: gate %u is not a 1..2-qubit fixed gate or a valid rotation", what, i);
            return nullptr;
        }
    }
    auto* a = new qm_adjoint();
    a->n = n;
    a->ne = ne;
    a->nparams = nparams;
    a->ngates = gate_count;
    a->build(b);
    return a;
}

void qm_adjoint_destroy(qm_adjoint* a) {
    if (!a) return;
    a->release();
    delete a;
}

void qm_adjoint_stats(const qm_adjoint* a, ITYPE* passes, ITYPE* gates) {
    ITYPE fs, fp, bs, bp;
    qm_adjoint_schedule(a, &fs, &fp, &bs, &bp);
    if (passes) *passes = fp + bp;
    if (gates) *gates = a ? (ITYPE)a->ngates : 0;
}

void qm_adjoint_schedule(const qm_adjoint* a, ITYPE* fwd_stages, ITYPE* fwd_passes, ITYPE* bwd_stages,
                         ITYPE* bwd_passes) {
    ITYPE fs = 0, fp = 0, bs = 0, bp = 0;
    if (a) {
        fs = a->fwd.stages.size();
        fp = a->fwd.passes.size();
        for (; bs < a->bwd.stages.size() && a->stage_grad0[bs] < a->ncols() / 3; ++bs) bp += a->bwd.stages[bs].npass;
    }
    if (fwd_stages) *fwd_stages = fs;
    if (fwd_passes) *fwd_passes = fp;
    if (bwd_stages) *bwd_stages = bs;
    if (bwd_passes) *bwd_passes = bp;
}

ITYPE qm_adjoint_workspace_bytes(const qm_adjoint* a, UINT batch) {
    if (!a) return 0;
    return 2 * a->state_bytes(batch) + a->fpool_bytes(batch) + a->bpool_bytes(batch) + a->part_bytes(batch) +
           a->sums_bytes(batch) + a->gvec_bytes(batch) + a->epart_bytes(batch) + 256;
}

int qm_adjoint_run(qm_adjoint* a, UINT batch, const double* theta, const ITYPE* bf, const ITYPE* pf, const UINT* rot,
                   const double* coefs, UINT nterms, double* energy, double* grad, void* workspace, void* stream,
                   unsigned dev) {
    const char* what = "qm_adjoint_run";
    if (!a || batch == 0 || batch > 65535 || !theta || !energy || !workspace || (nterms && (!bf || !pf || !rot || !coefs)) ||
        (a->nparams && !grad)) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null argument or batch outside 1..65535", what);
        return QM_ERR_INVALID_ARGUMENT;
    }
    for (UINT k = 0; k < nterms; ++k)
        if (((bf[k] | pf[k]) >> a->n) != 0) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: term %u acts beyond %u qubits", what, k, a->n);
            return QM_ERR_INVALID_ARGUMENT;
        }
    if (!use_device(dev)) return QM_ERR_HIP;
    hipStream_t st = stream_of(stream);
    if (!a->prepare(dev, what)) return QM_ERR_HIP;
    Scratch* sc = scratch_for(st);
    if (!sc) return QM_ERR_HIP;
    const u64 dim = 1ULL << a->ne;
    char* w = (char*)workspace;
    auto take = [&](u64 bytes) {
        char* p = w;
        w += bytes;
        return p;
    };
    double2* psi = (double2*)take(a->state_bytes(batch));
    double2* lam = (double2*)take(a->state_bytes(batch));
    double2* fpool = (double2*)take(a->fpool_bytes(batch));
    double2* bpool = (double2*)take(a->bpool_bytes(batch));
    double* partials = (double*)take(a->part_bytes(batch));
    double* sums = (double*)take(a->sums_bytes(batch));
    double* gvec = (double*)take(a->gvec_bytes(batch));
    double* epart = (double*)take(a->epart_bytes(batch));
    // the observable, grouped by bit-flip mask (groups and terms in the order given)
    std::vector<AdjGroup> groups;
    std::vector<AdjTerm> terms;
    {
        std::vector<bool> done(nterms, false);
        for (UINT k = 0; k < nterms; ++k) {
            if (done[k]) continue;
            AdjGroup g{bf[k], (u32)terms.size(), 0};
            for (UINT j = k; j < nterms; ++j)
                if (!done[j] && bf[j] == bf[k]) {
                    done[j] = true;
                    terms.push_back(AdjTerm{pf[j], rot[j], 0, coefs[j]});
                    ++g.nterm;
                }
            groups.push_back(g);
        }
    }
    const AdjGroup* dgroups = nullptr;
    const AdjTerm* dterms = nullptr;
    if (nterms) {
        dgroups = (const AdjGroup*)upload(sc, groups.data(), sizeof(AdjGroup) * groups.size());
        dterms = (const AdjTerm*)upload(sc, terms.data(), sizeof(AdjTerm) * terms.size());
        if (!dgroups || !dterms) return QM_ERR_HIP;
    }
    MatsArgs ma{a->d_factors, a->d_first, a->d_fixed, a->d_fwd_at, a->d_bwd_at, a->d_copies, a->d_copy_val,
                a->d_low, a->nops(), a->ncopy_f, a->ncopy_b, a->nparams, a->nocc(), (u32)a->fwd.pool.size(),
                (u32)a->bwd.pool.size()};
    const u32 nmat = a->nops() + a->ncopy_f + a->ncopy_b;
    if (nmat) k_adj_mats<<<dim3((nmat + 63) / 64, batch), 64, 0, st>>>(ma, theta, fpool, bpool, gvec);
    auto threads = [](u32 lq, u32 most) { return std::max(64u, std::min(most, (1u << lq) >> kAdjK)); };
    {
        const dim3 grid((u32)(1ULL << (a->ne - a->lqf)), batch);
        u32 first = 1;
        for (const DStage& sg : a->fwd.stages) {
            k_adj_fwd<<<grid, threads(a->lqf, kFwdThreads), sizeof(double2) << a->lqf, st>>>(
                psi, a->ne, a->lqf, first, sg, a->d_fpass, a->d_fsub, fpool, (u32)a->fwd.pool.size());
            first = 0;
        }
    }
    k_adj_hpsi<<<dim3(a->blocks_h(), batch), kHpsiThreads, 0, st>>>(psi, lam, dim, dgroups, (u32)groups.size(), dterms,
                                                                   epart);
    if (a->ncols()) {
        const dim3 grid(a->blocks_b(), batch);
        for (size_t c = 0; c + 1 < a->chunk0.size(); ++c) {
            const u32 first = a->stage_grad0[a->chunk0[c]], cols = 3 * (a->stage_grad0[a->chunk0[c + 1]] - first);
            if (cols == 0) continue;  // only stages behind the last rotation
            for (u32 s = a->chunk0[c]; s < a->chunk0[c + 1]; ++s) {
                if (a->stage_grad0[s] == a->ncols() / 3) break;  // no rotation is left: nothing more to differentiate
                k_adj_bwd<<<grid, threads(a->lqb, kBwdThreads), 2 * sizeof(double2) << a->lqb, st>>>(
                    psi, lam, a->ne, a->lqb, a->tiles_b(), a->bwd.stages[s], a->stage_grad0[s],
                    a->stage_grad0[s + 1] - a->stage_grad0[s], 3 * (a->stage_grad0[s] - first), a->d_bpass, a->d_bsub,
                    bpool, (u32)a->bwd.pool.size(), partials, cols);
            }
            k_adj_columns<<<dim3((cols + 15) / 16, batch), 256, 0, st>>>(partials, a->blocks_b(), cols, sums, a->ncols(),
                                                                         3 * first);
        }
    }
    k_adj_grad<<<dim3(std::max(1u, (a->nparams + 63) / 64), batch), 64, 0, st>>>(
        sums, a->ncols(), gvec, a->nocc(), a->d_par_first, a->d_par_occs, a->d_occ_col, a->d_occ_coef, a->nparams, grad,
        epart, a->blocks_h(), energy);
    if (!hip_ok(hipGetLastError(), what)) return QM_ERR_HIP;
    finish_update(st, what);
    return QM_OK;
}

}  // extern "C"
