// The tile engine shared by the batched / fused circuit executors and the
// adjoint gradients: a gate list is scheduled on the host into stages (gates whose
// qubits fit one window of a tile held in LDS) and, inside a stage, into passes
// (gates a thread applies to the 2^K amplitudes of K block qubits held in
// registers); the device half applies the passes of a stage to a tile in LDS.
// The scheme and its scheduling rule are described at the top of qm_batch.hip.
#pragma once

#include <algorithm>
#include <cmath>
#include <complex>
#include <vector>

#include "qm_internal.hpp"

namespace qm {
namespace {

using cd = std::complex<double>;

constexpr u32 kMaxLocal = 13;   // qubits resident in LDS
constexpr u32 kLowFixed = 4;    // qubits 0..3 are local in every stage (the executors; LOW below)
constexpr u32 kMinQubits = 4;   // smaller circuits run on 4 qubits (extra qubits stay |0>)

// Sub-operation kinds (low byte of DSub::type).
// LAYER: CZ gates, then one 2x2 matrix on each block bit of a mask.  type bits
//   8..11: the block-bit mask; bits 16..31: the sign pattern over the register
//   block of the CZs between two block bits; bit 15: a and m hold, for block
//   bit i, the mask of local positions outside the block that share a CZ with
//   it (16 bits each: a = M0 | M1 << 16, m = M2 | M3 << 16), so the sign of
//   register slot j changes with the parity of base & M_i where bit i of j is
//   set; bits 12..14: the number (<= 4) of CZs between two positions outside
//   the block, byte c of pairs = p | q << 4.
//   data: the matrices (4 complex each) of the mask's bits in ascending order.
// D2: 4x4 on block bits byte 0 / byte 1 of a; DK: 2^K x 2^K on the block;
// DIAG: diagonal on the m local positions in the bytes of a.
enum : u32 { SUB_LAYER = 0, SUB_D2 = 1, SUB_DK = 2, SUB_DIAG = 3 };
// bits 16 i .. 16 i + 15: the register-block indices j (< 16) with bit i set
constexpr u64 kBlockPatterns = 0xFF00F0F0CCCCAAAAull;
constexpr u32 kCzPairsMax = 4;

// Qubit lists are packed one byte per entry into 64-bit words so that the
// kernel indexes them with shifts (a runtime index into an array would put it
// in private memory).
struct DStage {
    u64 win[2];   // local bit LOW + i <-> qubit byte i of win (i < lq - LOW <= 10)
    u64 comp[4];  // tile bit i <-> qubit byte i of comp (i < n - lq <= 32)
    u32 npass, pass0;
};
__host__ __device__ __forceinline__ u32 byte_at(u64 w, u32 i) { return (u32)(w >> (8 * i)) & 0xffu; }
__host__ __forceinline__ void set_byte(u64& w, u32 i, u32 v) { w = (w & ~(0xffULL << (8 * i))) | ((u64)v << (8 * i)); }
struct DPass {
    unsigned char pos[4];  // block bits (local positions, ascending)
    u32 nsub, sub0;
    u32 flags;             // kPassHasDiag: a DIAG sub-operation (one register block per thread)
    unsigned short sbit[4];   // slot_of(1 << pos[i]), computed on the host
};
constexpr u32 kPassHasDiag = 1;
struct DSub {
    u32 type;
    u32 a;      // D2: block-bit indices (bytes); DIAG: local positions (bytes); LAYER: CZ masks
    u32 m;      // DIAG: qubit count; LAYER: CZ masks
    u32 data;   // offset into the complex pool
    u32 pairs;  // LAYER: CZs between two positions outside the block
    u32 grad0;  // LAYER: position in Flat::grads of the first matrix in gmask
    u32 gmask;  // LAYER: block bits whose matrix belongs to an operation with grad set
    u32 pad;
};
struct DTerm {
    u64 bf, pf;
    u32 rot, pad;
    double coef;
};

struct HOp {
    u32 type;  // 0 dense, 1 diag, 2 cz
    std::vector<u32> q;
    std::vector<cd> m;
    long id = -1;       // the caller's number of a single-qubit dense operation (see Flat::mats)
    bool grad = false;  // listed in Flat::grads
    u64 mask() const {
        u64 r = 0;
        for (u32 x : q) r |= 1ULL << x;
        return r;
    }
};
struct HCirc {
    u32 n = 0;  // as given
    u32 ne = 0; // as run (>= kMinQubits)
    std::vector<HOp> ops;
    std::vector<DTerm> terms;
};


__host__ __device__ __forceinline__ u32 fold3(u32 x) { return ((x >> 3) ^ (x >> 6) ^ (x >> 9) ^ (x >> 12)) & 7u; }
__host__ __device__ __forceinline__ u32 slot_of(u32 x) { return x ^ fold3(x); }

// (x, y) <- (m0 x + m1 y, m2 x + m3 y), complex, updated in place; the matrix
// entries are wave-uniform (scalar registers).  Written as one asm block so the
// four results land in the registers of the four inputs: the sub-operation loop
// of run_passes then keeps the register block at fixed registers across all
// sub-operation kinds instead of copying it at every merge point.  The last
// reader of each input writes a result into it (x.re holds the x.re chain from
// its 4th op on), so three temporaries suffice.
__device__ __forceinline__ void pair_update(double2& x, double2& y, const double2 m0, const double2 m1,
                                            const double2 m2, const double2 m3) {
    double tb, tc, td;
    asm("v_mul_f64 %[tb], %[m0i], %[xr]\n\t"          // B = x'.im
        "v_mul_f64 %[tc], %[m2r], %[xr]\n\t"          // C = y'.re
        "v_mul_f64 %[td], %[m2i], %[xr]\n\t"          // D = y'.im
        "v_mul_f64 %[xr], %[m0r], %[xr]\n\t"          // A = x'.re
        "v_fma_f64 %[xr], -%[m0i], %[xi], %[xr]\n\t"
        "v_fma_f64 %[tb], %[m0r], %[xi], %[tb]\n\t"
        "v_fma_f64 %[tc], -%[m2i], %[xi], %[tc]\n\t"
        "v_fma_f64 %[td], %[m2r], %[xi], %[td]\n\t"
        "v_fma_f64 %[xr], %[m1r], %[yr], %[xr]\n\t"
        "v_fma_f64 %[tb], %[m1i], %[yr], %[tb]\n\t"
        "v_fma_f64 %[tc], %[m3r], %[yr], %[tc]\n\t"
        "v_fma_f64 %[td], %[m3i], %[yr], %[td]\n\t"
        "v_fma_f64 %[xi], %[m1r], %[yi], %[tb]\n\t"
        "v_fma_f64 %[yr], -%[m3i], %[yi], %[tc]\n\t"
        "v_fma_f64 %[xr], -%[m1i], %[yi], %[xr]\n\t"
        "v_fma_f64 %[yi], %[m3r], %[yi], %[td]"
        : [xr] "+v"(x.x), [xi] "+v"(x.y), [yr] "+v"(y.x), [yi] "+v"(y.y), [tb] "=&v"(tb), [tc] "=&v"(tc),
          [td] "=&v"(td)
        : [m0r] "s"(m0.x), [m0i] "s"(m0.y), [m1r] "s"(m1.x), [m1i] "s"(m1.y), [m2r] "s"(m2.x), [m2i] "s"(m2.y),
          [m3r] "s"(m3.x), [m3i] "s"(m3.y));
}

// v <- v * z, complex, in place.
__device__ __forceinline__ void cmul_inplace(double2& v, const double2 z) {
    double t;
    asm("v_mul_f64 %[t], %[vr], %[zi]\n\t"
        "v_mul_f64 %[vr], %[vr], %[zr]\n\t"
        "v_fma_f64 %[vr], -%[vi], %[zi], %[vr]\n\t"
        "v_fma_f64 %[vi], %[vi], %[zr], %[t]"
        : [vr] "+v"(v.x), [vi] "+v"(v.y), [t] "=&v"(t)
        : [zr] "v"(z.x), [zi] "v"(z.y));
}

// Two independent pair updates interleaved instruction by instruction, so a
// dependent FMA follows its producer 8 instructions later (pair_update alone:
// 4), which keeps the FP64 pipeline busy with only two waves per SIMD.
__device__ __forceinline__ void pair_update2(double2& x0, double2& y0, double2& x1, double2& y1, const double2 m0,
                                             const double2 m1, const double2 m2, const double2 m3) {
    double tb0, tc0, td0, tb1, tc1, td1;
    asm("v_mul_f64 %[tb0], %[m0i], %[xr0]\n\t"
        "v_mul_f64 %[tb1], %[m0i], %[xr1]\n\t"
        "v_mul_f64 %[tc0], %[m2r], %[xr0]\n\t"
        "v_mul_f64 %[tc1], %[m2r], %[xr1]\n\t"
        "v_mul_f64 %[td0], %[m2i], %[xr0]\n\t"
        "v_mul_f64 %[td1], %[m2i], %[xr1]\n\t"
        "v_mul_f64 %[xr0], %[m0r], %[xr0]\n\t"
        "v_mul_f64 %[xr1], %[m0r], %[xr1]\n\t"
        "v_fma_f64 %[xr0], -%[m0i], %[xi0], %[xr0]\n\t"
        "v_fma_f64 %[xr1], -%[m0i], %[xi1], %[xr1]\n\t"
        "v_fma_f64 %[tb0], %[m0r], %[xi0], %[tb0]\n\t"
        "v_fma_f64 %[tb1], %[m0r], %[xi1], %[tb1]\n\t"
        "v_fma_f64 %[tc0], -%[m2i], %[xi0], %[tc0]\n\t"
        "v_fma_f64 %[tc1], -%[m2i], %[xi1], %[tc1]\n\t"
        "v_fma_f64 %[td0], %[m2r], %[xi0], %[td0]\n\t"
        "v_fma_f64 %[td1], %[m2r], %[xi1], %[td1]\n\t"
        "v_fma_f64 %[xr0], %[m1r], %[yr0], %[xr0]\n\t"
        "v_fma_f64 %[xr1], %[m1r], %[yr1], %[xr1]\n\t"
        "v_fma_f64 %[tb0], %[m1i], %[yr0], %[tb0]\n\t"
        "v_fma_f64 %[tb1], %[m1i], %[yr1], %[tb1]\n\t"
        "v_fma_f64 %[tc0], %[m3r], %[yr0], %[tc0]\n\t"
        "v_fma_f64 %[tc1], %[m3r], %[yr1], %[tc1]\n\t"
        "v_fma_f64 %[td0], %[m3i], %[yr0], %[td0]\n\t"
        "v_fma_f64 %[td1], %[m3i], %[yr1], %[td1]\n\t"
        "v_fma_f64 %[xi0], %[m1r], %[yi0], %[tb0]\n\t"
        "v_fma_f64 %[xi1], %[m1r], %[yi1], %[tb1]\n\t"
        "v_fma_f64 %[yr0], -%[m3i], %[yi0], %[tc0]\n\t"
        "v_fma_f64 %[yr1], -%[m3i], %[yi1], %[tc1]\n\t"
        "v_fma_f64 %[xr0], -%[m1i], %[yi0], %[xr0]\n\t"
        "v_fma_f64 %[xr1], -%[m1i], %[yi1], %[xr1]\n\t"
        "v_fma_f64 %[yi0], %[m3r], %[yi0], %[td0]\n\t"
        "v_fma_f64 %[yi1], %[m3r], %[yi1], %[td1]"
        : [xr0] "+v"(x0.x), [xi0] "+v"(x0.y), [yr0] "+v"(y0.x), [yi0] "+v"(y0.y), [xr1] "+v"(x1.x),
          [xi1] "+v"(x1.y), [yr1] "+v"(y1.x), [yi1] "+v"(y1.y), [tb0] "=&v"(tb0), [tc0] "=&v"(tc0),
          [td0] "=&v"(td0), [tb1] "=&v"(tb1), [tc1] "=&v"(tc1), [td1] "=&v"(td1)
        : [m0r] "s"(m0.x), [m0i] "s"(m0.y), [m1r] "s"(m1.x), [m1i] "s"(m1.y), [m2r] "s"(m2.x), [m2i] "s"(m2.y),
          [m3r] "s"(m3.x), [m3i] "s"(m3.y));
}

// One 2x2 matrix on block bit P of each of the G register blocks of a thread.
// With two blocks, the pair updates interleave pair q of block 0 with pair q of
// block 1; with one block, pairs q and q + 1.
template <int K, int P, int G>
__device__ __forceinline__ void sub_d1(double2 (&v)[G][1 << K], const double2* mp) {
    const double2 m0 = mp[0], m1 = mp[1], m2 = mp[2], m3 = mp[3];
    // the 2^(K-1) pairs (j, j | 2^P)
    constexpr int NP = 1 << (K - 1);
    auto pair_j = [](int q) { return ((q >> P) << (P + 1)) | (q & ((1 << P) - 1)); };
    if constexpr (G == 2) {
#pragma unroll
        for (int q = 0; q < NP; ++q)
            pair_update2(v[0][pair_j(q)], v[0][pair_j(q) | (1 << P)], v[1][pair_j(q)], v[1][pair_j(q) | (1 << P)], m0,
                         m1, m2, m3);
    } else {
#pragma unroll
        for (int q = 0; q < NP; q += 2)
            pair_update2(v[0][pair_j(q)], v[0][pair_j(q) | (1 << P)], v[0][pair_j(q + 1)],
                         v[0][pair_j(q + 1) | (1 << P)], m0, m1, m2, m3);
    }
}

template <int K, int P0, int P1>
__device__ __forceinline__ void sub_d2(double2* v, const double2* mp) {
    double2 m[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) m[i] = mp[i];
#pragma unroll
    for (int j = 0; j < (1 << K); ++j) {
        if (j & ((1 << P0) | (1 << P1))) continue;
        const double2 i0 = v[j], i1 = v[j | (1 << P0)], i2 = v[j | (1 << P1)], i3 = v[j | (1 << P0) | (1 << P1)];
        v[j] = cmac(cmac(cmac(cmul(m[0], i0), m[1], i1), m[2], i2), m[3], i3);
        v[j | (1 << P0)] = cmac(cmac(cmac(cmul(m[4], i0), m[5], i1), m[6], i2), m[7], i3);
        v[j | (1 << P1)] = cmac(cmac(cmac(cmul(m[8], i0), m[9], i1), m[10], i2), m[11], i3);
        v[j | (1 << P0) | (1 << P1)] = cmac(cmac(cmac(cmul(m[12], i0), m[13], i1), m[14], i2), m[15], i3);
    }
}

template <int K>
__device__ __forceinline__ void sub_dk(double2* v, const double2* mp) {
    constexpr int D = 1 << K;
    double2 out[D];
#pragma unroll
    for (int r = 0; r < D; ++r) {
        double2 acc = cmul(mp[r * D], v[0]);
#pragma unroll
        for (int c = 1; c < D; ++c) acc = cmac(acc, mp[r * D + c], v[c]);
        out[r] = acc;
    }
#pragma unroll
    for (int r = 0; r < D; ++r) v[r] = out[r];
}

#define QM_D2_CASE(A, B) \
    case (A) * 4 + (B):  \
        if constexpr (K > (A) && K > (B)) sub_d2<K, A, B>(v, mp); \
        break;
template <int K>
__device__ __forceinline__ void apply_d2(double2* v, u32 p0, u32 p1, const double2* mp) {
    switch (p0 * 4 + p1) {
        QM_D2_CASE(0, 1) QM_D2_CASE(0, 2) QM_D2_CASE(0, 3)
        QM_D2_CASE(1, 0) QM_D2_CASE(1, 2) QM_D2_CASE(1, 3)
        QM_D2_CASE(2, 0) QM_D2_CASE(2, 1) QM_D2_CASE(2, 3)
        QM_D2_CASE(3, 0) QM_D2_CASE(3, 1) QM_D2_CASE(3, 2)
        default: break;
    }
}
#undef QM_D2_CASE

// hi_tab[j] = global offset of local index j << LOW (the window qubits LOW.. of the
// stage).  TI = u32 holds offsets below 2^32 (states of at most 32 qubits);
// larger states use u64.
template <u32 LOW = kLowFixed, typename TI>
__device__ __forceinline__ void build_hi_tab(TI* hi_tab, u32 lq, const DStage& sg) {
    const u64 win0 = sg.win[0], win1 = sg.win[1];
    for (u32 j = threadIdx.x; j < (1u << (lq - LOW)); j += blockDim.x) {
        TI o = 0;
        for (u32 i = 0; i + LOW < lq; ++i) o |= (TI)((j >> i) & 1u) << byte_at(i < 8 ? win0 : win1, i & 7);
        hi_tab[j] = o;
    }
}

// global index of the first amplitude of tile t (tile bits deposited on the non-window qubits)
__device__ __forceinline__ u64 tile_base(u64 t, u32 tl, const DStage& sg) {
    const u64 c0 = sg.comp[0], c1 = sg.comp[1], c2 = sg.comp[2], c3 = sg.comp[3];
    u64 tb = 0;
    for (u32 i = 0; i < tl; ++i) {
        const u64 w = i < 8 ? c0 : i < 16 ? c1 : i < 24 ? c2 : c3;
        tb |= ((t >> i) & 1ULL) << byte_at(w, i & 7);
    }
    return tb;
}

template <u32 LOW = kLowFixed, typename TI>
__device__ __forceinline__ u64 tile_index(u64 tb, const TI* hi_tab, u32 i) {
    return tb + hi_tab[i >> LOW] + (i & ((1u << LOW) - 1));
}

// The signs that the CZ gates of a LAYER give a register block with block base
// `base` (local index with zeros at the block positions): bit j of the result set
// means that amplitude j changes sign.  base is zero at the block positions, so a
// local position p outside the block is (base >> p) & 1 for the whole block.
template <int K>
__device__ __forceinline__ u32 layer_signs(const DSub& sub, u32 base) {
    u32 sgn = sub.type >> 16;
    if (sub.type & 0x8000u) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const u32 mi = ((i < 2 ? sub.a : sub.m) >> (16 * (i & 1))) & 0xffffu;
            constexpr u32 kPat[4] = {(u32)(kBlockPatterns & 0xffffu), (u32)((kBlockPatterns >> 16) & 0xffffu),
                                     (u32)((kBlockPatterns >> 32) & 0xffffu), (u32)(kBlockPatterns >> 48)};
            sgn ^= (0u - ((u32)__popc(base & mi) & 1u)) & kPat[i];
        }
    }
    const u32 npair = (sub.type >> 12) & 7u;
    for (u32 c = 0; c < npair; ++c) {
        const u32 w = sub.pairs >> (8 * c), p0 = w & 15u, p1 = (w >> 4) & 15u;
        sgn ^= 0u - ((base >> p0) & (base >> p1) & 1u);
    }
    return sgn;
}
// flips the sign bits of both components of v[j] where bit j of sgn is set
template <int K>
__device__ __forceinline__ void flip_signs(double2 (&v)[1 << K], u32 sgn) {
#pragma unroll
    for (int j = 0; j < (1 << K); ++j) {
        const int f = (int)((sgn << (31 - j)) & 0x80000000u);
        v[j].x = __hiloint2double(__double2hiint(v[j].x) ^ f, __double2loint(v[j].x));
        v[j].y = __hiloint2double(__double2hiint(v[j].y) ^ f, __double2loint(v[j].y));
    }
}

// One LAYER sub-operation on the G register blocks of a thread, block g with
// block base base[g].  The sub-operation is decoded once for all blocks.
template <int K, int G>
__device__ __forceinline__ void apply_layer(double2 (&v)[G][1 << K], const DSub& sub, const u32 (&base)[G],
                                            const double2* __restrict__ pool) {
    const u32 d1 = (sub.type >> 8) & 15u;
    if (sub.type >> 12) {
        u32 sgn[G];
#pragma unroll
        for (int g = 0; g < G; ++g) sgn[g] = layer_signs<K>(sub, base[g]);
#pragma unroll
        for (int g = 0; g < G; ++g) flip_signs<K>(v[g], sgn[g]);
    }
    const double2* mp = pool + sub.data;
    if (d1 & 1u) {
        sub_d1<K, 0, G>(v, mp);
        mp += 4;
    }
    if (d1 & 2u) {
        sub_d1<K, 1, G>(v, mp);
        mp += 4;
    }
    if constexpr (K > 2)
        if (d1 & 4u) {
            sub_d1<K, 2, G>(v, mp);
            mp += 4;
        }
    if constexpr (K > 3)
        if (d1 & 8u) sub_d1<K, 3, G>(v, mp);
}

// The sub-operations of one pass on the G register blocks of groups gi0,
// gi0 + T, ..., read from and written back to LDS.  slot_of is linear over
// GF(2), so the slot of base | off[j] is slot_of(base) ^ (XOR of sbit[i] over
// the bits i of j): each lane forms its 2^K slots from the K per-bit offsets
// (the empty asm keeps every partial XOR in a vector register, so the compiler
// does not form the 2^K uniform combinations in scalar registers, which spill).
// WIDE = false: only LAYER and D2 sub-operations occur.
template <int K, u32 T, int G, bool WIDE = true>
__device__ __forceinline__ void pass_groups(double2* st, const DPass& ps, const u32 (&sbit)[K], u32 gi0,
                                            const DSub* __restrict__ subs, const double2* __restrict__ pool) {
    constexpr int D = 1 << K;
    u32 base[G], slot[G][D];
    double2 v[G][D];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        u32 b = gi0 + (u32)g * T;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const u32 q = ps.pos[i];
            b = (b & ((1u << q) - 1)) | ((b >> q) << (q + 1));
        }
        base[g] = b;
        slot[g][0] = slot_of(b);
#pragma unroll
        for (int j = 1; j < D; ++j) {
            const int lb = __builtin_ctz(j);
            slot[g][j] = slot[g][j & (j - 1)] ^ sbit[lb];
            // one block per thread: keep the chain per lane (see above); two
            // blocks: the 2^K uniform offsets are formed once and shared, which
            // costs fewer vector registers where both blocks are live
            if constexpr (G == 1) asm volatile("" : "+v"(slot[g][j]));
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int j = 0; j < D; ++j) v[g][j] = st[slot[g][j]];
    // LAYER sub-operations run in an inner loop of their own and update the
    // register blocks in place, so the blocks stay at fixed registers there;
    // the other kinds are handled between runs of LAYERs.
    u32 k = 0;
    while (k < ps.nsub) {
        DSub sub = subs[ps.sub0 + k];
        while ((sub.type & 0xffu) == SUB_LAYER) {
            apply_layer<K, G>(v, sub, base, pool);
            if (++k == ps.nsub) break;
            sub = subs[ps.sub0 + k];
        }
        if (k == ps.nsub) break;
        const u32 kind = sub.type & 0xffu;
        const double2* mp = pool + sub.data;
        if (kind == SUB_D2) {
#pragma unroll
            for (int g = 0; g < G; ++g) apply_d2<K>(v[g], byte_at(sub.a, 0), byte_at(sub.a, 1), mp);
        } else if (WIDE && kind == SUB_DK) {
#pragma unroll
            for (int g = 0; g < G; ++g) sub_dk<K>(v[g], mp);
        } else if (WIDE && G == 1 && kind == SUB_DIAG) {
            // (passes with a DIAG run with one block per thread: the per-lane
            // reads of the diagonal for two blocks exhaust the registers)
            // bit i of the diagonal index: local position p_i, i.e. bit p_i of
            // base or, for a block position, bit j of the block pattern
            u32 pat[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u32 p = byte_at(sub.a, i);
                u32 pt = 0;
#pragma unroll
                for (int b = 0; b < K; ++b) pt |= (ps.pos[b] == p) ? (u32)(kBlockPatterns >> (16 * b)) & 0xffffu : 0u;
                pat[i] = i < (int)sub.m ? pt : 0u;
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                u32 tbit[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) tbit[i] = i < (int)sub.m ? (base[g] >> byte_at(sub.a, i)) & 1u : 0u;
#pragma unroll
                for (int j = 0; j < D; ++j) {
                    u32 idx = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) idx |= ((tbit[i] | (pat[i] >> j)) & 1u) << i;
                    cmul_inplace(v[g][j], mp[idx]);
                }
            }
        }
        ++k;
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int j = 0; j < D; ++j) st[slot[g][j]] = v[g][j];
}

// Applies passes [pass0, pass0 + npass) to the 2^lq amplitudes in LDS with a
// work-group of T threads (of at most T if it has fewer groups than T); ends with a barrier after every pass.  With G = 2
// and exactly 2 T groups of 2^K amplitudes, every thread holds two register
// blocks and decodes each sub-operation once for both.
template <int K, u32 T, int G, bool WIDE = true>
__device__ __forceinline__ void run_passes(double2* st, u32 lq, const DPass* __restrict__ passes, u32 pass0,
                                           u32 npass, const DSub* __restrict__ subs,
                                           const double2* __restrict__ pool) {
    constexpr int D = 1 << K;
    const u32 ngroups = (1u << lq) >> K;
    for (u32 p = 0; p < npass; ++p) {
        const DPass ps = passes[pass0 + p];
        u32 sbit[K];
#pragma unroll
        for (int i = 0; i < K; ++i) sbit[i] = ps.sbit[i];
        if (G == 2 && ngroups == 2 * T && !(ps.flags & kPassHasDiag)) {
            pass_groups<K, T, G, WIDE>(st, ps, sbit, threadIdx.x, subs, pool);
        } else if (ngroups == T) {
            pass_groups<K, T, 1, WIDE>(st, ps, sbit, threadIdx.x, subs, pool);
        } else {
            for (u32 g = threadIdx.x; g < ngroups; g += blockDim.x)
                pass_groups<K, T, 1, WIDE>(st, ps, sbit, g, subs, pool);
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ host side
void mat_mul(const std::vector<cd>& a, const std::vector<cd>& b, std::vector<cd>& out, int d) {
    out.assign((size_t)d * d, 0.0);
    for (int i = 0; i < d; ++i)
        for (int k = 0; k < d; ++k)
            for (int j = 0; j < d; ++j) out[i * d + j] += a[i * d + k] * b[k * d + j];
}

// Schedules one circuit; appends to the flat arrays.
struct Flat {
    std::vector<DStage> stages;
    std::vector<DPass> passes;
    std::vector<DSub> subs;
    std::vector<double2> pool;
    // (id, pool offset) of every matrix of an operation with an id, and the ids of
    // those with grad set, both in the order in which the passes apply them
    std::vector<std::pair<long, u32>> mats;
    std::vector<long> grads;
};

u32 pool_put(Flat& f, const std::vector<cd>& m) {
    const u32 off = (u32)f.pool.size();
    for (const cd& z : m) f.pool.push_back(make_double2(z.real(), z.imag()));
    return off;
}

// Passes of one stage: ops (already in local positions) -> DPass/DSub.
void schedule_passes(Flat& f, std::vector<HOp> ops, u32 lq, u32 K, DStage& sg) {
    sg.pass0 = (u32)f.passes.size();
    sg.npass = 0;
    std::vector<bool> done(ops.size(), false);
    size_t left = ops.size();
    while (left > 0) {
        u64 blocked = 0, block = 0;
        std::vector<size_t> sel;
        for (size_t i = 0; i < ops.size(); ++i) {
            if (done[i]) continue;
            const HOp& o = ops[i];
            const u64 m = o.mask();
            if (m & blocked) {
                blocked |= m;
                continue;
            }
            if (o.type != 0) {
                sel.push_back(i);
                continue;
            }
            if ((u32)__builtin_popcountll(block | m) <= K) {
                block |= m;
                sel.push_back(i);
            } else {
                blocked |= m;
            }
        }
        // pad the block to K local positions
        for (u32 p = 0; p < lq && (u32)__builtin_popcountll(block) < K; ++p) block |= 1ULL << p;
        DPass ps{};
        u32 bpos[4] = {0, 0, 0, 0};
        {
            u32 k = 0;
            for (u32 p = 0; p < lq; ++p)
                if ((block >> p) & 1) bpos[k++] = p;
        }
        for (u32 i = 0; i < 4; ++i) ps.pos[i] = (unsigned char)bpos[i];
        for (u32 i = 0; i < K; ++i) ps.sbit[i] = (unsigned short)slot_of(1u << bpos[i]);
        ps.sub0 = (u32)f.subs.size();
        auto bit_of = [&](u32 p) -> u32 {
            for (u32 i = 0; i < K; ++i)
                if (bpos[i] == p) return i;
            return 0;
        };
        // Consecutive CZ gates, then consecutive single-qubit matrices on distinct
        // block bits (these commute with each other), become one LAYER.
        std::vector<const HOp*> pend_d1(K, nullptr);
        u32 d1mask = 0, cz_const = 0, npair = 0, pairs = 0;
        u32 czmask[4] = {0, 0, 0, 0};
        bool cz_any = false;
        auto flush = [&]() {
            if (d1mask == 0 && !cz_any) return;
            DSub sb{};
            const bool masks = (czmask[0] | czmask[1] | czmask[2] | czmask[3]) != 0;
            sb.type = SUB_LAYER | (d1mask << 8) | (npair << 12) | (masks ? 0x8000u : 0u) | (cz_const << 16);
            sb.a = czmask[0] | (czmask[1] << 16);
            sb.m = czmask[2] | (czmask[3] << 16);
            sb.pairs = pairs;
            sb.data = (u32)f.pool.size();
            sb.grad0 = (u32)f.grads.size();
            for (u32 b = 0; b < K; ++b) {
                if (!pend_d1[b]) continue;
                const u32 off = pool_put(f, pend_d1[b]->m);
                if (pend_d1[b]->id >= 0) f.mats.emplace_back(pend_d1[b]->id, off);
                if (pend_d1[b]->grad) {
                    sb.gmask |= 1u << b;
                    f.grads.push_back(pend_d1[b]->id);
                }
            }
            f.subs.push_back(sb);
            std::fill(pend_d1.begin(), pend_d1.end(), nullptr);
            d1mask = 0;
            cz_const = 0;
            npair = 0;
            pairs = 0;
            std::fill(czmask, czmask + 4, 0u);
            cz_any = false;
        };
        const u32 jmask = (1u << (1u << K)) - 1;
        auto add_cz = [&](u32 p0, u32 p1) {
            const bool in0 = (block >> p0) & 1, in1 = (block >> p1) & 1;
            if (in0 && in1) {
                cz_const ^= (u32)(kBlockPatterns >> (16 * bit_of(p0))) & (u32)(kBlockPatterns >> (16 * bit_of(p1))) &
                            jmask;
            } else if (in0 || in1) {
                czmask[bit_of(in0 ? p0 : p1)] ^= 1u << (in0 ? p1 : p0);
            } else {
                if (npair == kCzPairsMax) flush();
                pairs |= (p0 | (p1 << 4)) << (8 * npair);
                ++npair;
            }
            cz_any = true;
        };
        for (size_t i : sel) {
            const HOp& o = ops[i];
            done[i] = true;
            --left;
            if (o.type == 2) {
                if (d1mask) flush();
                add_cz(o.q[0], o.q[1]);
                continue;
            }
            if (o.type == 0 && o.q.size() == 1) {
                const u32 b = bit_of(o.q[0]);
                if ((d1mask >> b) & 1) flush();
                pend_d1[b] = &o;
                d1mask |= 1u << b;
                continue;
            }
            flush();
            DSub sb{};
            if (o.type == 1) {
                ps.flags |= kPassHasDiag;
                sb.type = SUB_DIAG;
                sb.m = (u32)o.q.size();
                for (size_t k = 0; k < o.q.size(); ++k) sb.a |= o.q[k] << (8 * k);
                sb.data = pool_put(f, o.m);
            } else if (o.q.size() == 2) {
                sb.type = SUB_D2;
                sb.a = bit_of(o.q[0]) | (bit_of(o.q[1]) << 8);
                sb.data = pool_put(f, o.m);
            } else {
                // embed into the K block bits (ascending) with the identity elsewhere
                const u32 k = (u32)o.q.size(), D = 1u << K;
                std::vector<u32> bits(k);
                u32 omask = 0;
                for (u32 t = 0; t < k; ++t) {
                    bits[t] = bit_of(o.q[t]);
                    omask |= 1u << bits[t];
                }
                std::vector<cd> M((size_t)D * D, 0.0);
                for (u32 col = 0; col < D; ++col) {
                    u32 x = 0;
                    for (u32 t = 0; t < k; ++t) x |= ((col >> bits[t]) & 1u) << t;
                    for (u32 y = 0; y < (1u << k); ++y) {
                        u32 row = col & ~omask;
                        for (u32 t = 0; t < k; ++t) row |= ((y >> t) & 1u) << bits[t];
                        M[(size_t)row * D + col] += o.m[(size_t)y * (1u << k) + x];
                    }
                }
                sb.type = SUB_DK;
                sb.data = pool_put(f, M);
            }
            f.subs.push_back(sb);
        }
        flush();
        ps.nsub = (u32)f.subs.size() - ps.sub0;
        f.passes.push_back(ps);
        ++sg.npass;
    }
}

// Stages (windows of lq_cap qubits including 0..3) for circuits above lq_cap
// qubits; a single identity stage otherwise.  Returns the number of stages appended.
// `low`: the qubits below it are in every window.  `max_grads`: a stage takes at
// most that many operations with grad set.
u32 schedule_circuit(Flat& f, const HCirc& c, u32 K, u32 lq_cap = kMaxLocal, u32 low_fixed = kLowFixed,
                     size_t max_grads = ~size_t(0)) {
    const u32 n = c.ne, lq = std::min(n, lq_cap);
    if (n <= lq_cap && max_grads == ~size_t(0)) {
        DStage sg{};
        for (u32 i = 0; i + low_fixed < lq; ++i) set_byte(sg.win[i >> 3], i & 7, low_fixed + i);
        schedule_passes(f, c.ops, lq, K, sg);
        f.stages.push_back(sg);
        return 1;
    }
    std::vector<bool> done(c.ops.size(), false);
    size_t left = c.ops.size();
    u32 count = 0;
    const u64 low = (1ULL << low_fixed) - 1;
    while (left > 0) {
        u64 win = low, blocked = 0;
        size_t grads = 0;
        std::vector<size_t> sel;
        for (size_t i = 0; i < c.ops.size(); ++i) {
            if (done[i]) continue;
            const u64 m = c.ops[i].mask();
            if (m & blocked) {
                blocked |= m;
                continue;
            }
            if ((u32)__builtin_popcountll(win | m) <= lq && (!c.ops[i].grad || grads < max_grads)) {
                win |= m;
                grads += c.ops[i].grad ? 1 : 0;
                sel.push_back(i);
            } else {
                blocked |= m;
            }
        }
        for (u32 q = 0; q < n && (u32)__builtin_popcountll(win) < lq; ++q) win |= 1ULL << q;
        DStage sg{};
        u32 local_of[64];
        u32 wi = 0, ci = 0;
        for (u32 q = 0; q < n; ++q) {
            if (q < low_fixed) {
                local_of[q] = q;
            } else if ((win >> q) & 1) {
                local_of[q] = low_fixed + wi;
                set_byte(sg.win[wi >> 3], wi & 7, q);
                ++wi;
            } else {
                set_byte(sg.comp[ci >> 3], ci & 7, q);
                ++ci;
            }
        }
        std::vector<HOp> ops;
        ops.reserve(sel.size());
        for (size_t i : sel) {
            HOp o = c.ops[i];
            for (u32& q : o.q) q = local_of[q];
            ops.push_back(std::move(o));
            done[i] = true;
            --left;
        }
        schedule_passes(f, ops, lq, K, sg);
        f.stages.push_back(sg);
        ++count;
    }
    if (count == 0) {  // a circuit without gates still needs one stage to initialise |0>
        DStage sg{};
        u32 wi = 0, ci = 0;
        for (u32 q = low_fixed; q < n; ++q) {
            if (wi + low_fixed < lq) {
                set_byte(sg.win[wi >> 3], wi & 7, q);
                ++wi;
            } else {
                set_byte(sg.comp[ci >> 3], ci & 7, q);
                ++ci;
            }
        }
        sg.npass = 0;
        sg.pass0 = (u32)f.passes.size();
        f.stages.push_back(sg);
        count = 1;
    }
    return count;
}

// Gates in the C ABI form -> internal ops, with consecutive single-qubit dense /
// diagonal gates on the same qubit multiplied together.
// Appends o; a single-qubit dense / diagonal gate is fused into the previous
// op on its qubit when that is one too (last[q]: index of the last op on q).
void push_op(HCirc& c, std::vector<long>& last, HOp o) {
    if (o.q.size() == 1 && o.type != 2) {
        const long p = last[o.q[0]];
        if (p >= 0 && c.ops[p].q.size() == 1 && c.ops[p].type != 2) {
            HOp& prev = c.ops[p];
            auto full = [](const HOp& h) {
                if (h.type == 0) return h.m;
                return std::vector<cd>{h.m[0], 0.0, 0.0, h.m[1]};
            };
            if (prev.type == 1 && o.type == 1) {
                prev.m[0] *= o.m[0];
                prev.m[1] *= o.m[1];
            } else {
                std::vector<cd> prod;
                mat_mul(full(o), full(prev), prod, 2);  // new after old
                prev.m = prod;
                prev.type = 0;
            }
            return;
        }
    }
    c.ops.push_back(std::move(o));
    for (u32 q : c.ops.back().q) last[q] = (long)c.ops.size() - 1;
}

bool convert_gates(u32 n, const qm_batch_gate* gates, UINT gate_count, HCirc& c, const char* what) {
    c.n = n;
    c.ne = std::max<u32>(n, kMinQubits);
    std::vector<long> last(c.ne, -1);  // last op touching each qubit
    for (UINT gi = 0; gi < gate_count; ++gi) {
        const qm_batch_gate& g = gates[gi];
        const u32 k = g.qubit_count;
        const bool two = g.kind == QM_BATCH_CZ || g.kind == QM_BATCH_CNOT;
        if (g.kind > QM_BATCH_CNOT || k < 1 || k > 4 || (two && k != 2)) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: gate %u: kind %u with %u qubits is not supported", what, gi, g.kind, k);
            return false;
        }
        u64 mask = 0;
        for (u32 i = 0; i < k; ++i) {
            if (g.qubits[i] >= n || ((mask >> g.qubits[i]) & 1)) {
                set_error(QM_ERR_INVALID_ARGUMENT, "%s: gate %u: qubit %u out of range or repeated", what, gi, g.qubits[i]);
                return false;
            }
            mask |= 1ULL << g.qubits[i];
        }
        if ((g.kind == QM_BATCH_DENSE || g.kind == QM_BATCH_DIAG) && !g.matrix) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: gate %u: null matrix", what, gi);
            return false;
        }
        if (g.kind == QM_BATCH_CNOT) {
            // CNOT(c, t) = H_t CZ(c, t) H_t; the Hadamards fuse into the
            // single-qubit gates next to them on t
            const double h = 0.70710678118654752440;
            HOp hd;
            hd.type = 0;
            hd.q = {g.qubits[1]};
            hd.m = {h, h, h, -h};
            HOp cz;
            cz.type = 2;
            cz.q = {g.qubits[0], g.qubits[1]};
            push_op(c, last, hd);
            push_op(c, last, std::move(cz));
            push_op(c, last, std::move(hd));
            continue;
        }
        HOp o;
        o.q.assign(g.qubits, g.qubits + k);
        const u32 d = 1u << k;
        if (g.kind == QM_BATCH_CZ) {
            o.type = 2;
        } else if (g.kind == QM_BATCH_DIAG) {
            o.type = 1;
            for (u32 i = 0; i < d; ++i) o.m.push_back(cd(g.matrix[i].re, g.matrix[i].im));
        } else {
            o.type = 0;
            for (u32 i = 0; i < d * d; ++i) o.m.push_back(cd(g.matrix[i].re, g.matrix[i].im));
        }
        push_op(c, last, std::move(o));
    }
    return true;
}

}  // namespace
}  // namespace qm
