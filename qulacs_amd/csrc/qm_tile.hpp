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
// Host-side products of gate matrices are formed with 64 mantissa bits, so that a merged or
// factored matrix carries little more than the rounding of its final entries.
using cx = std::complex<long double>;
inline cx mul(const cx& a, const cx& b) {  // without the C library's checks for infinities
    return cx(a.real() * b.real() - a.imag() * b.imag(), a.real() * b.imag() + a.imag() * b.real());
}
inline cx quot(const cx& a, const cx& b) { return mul(a, std::conj(b)) / std::norm(b); }

constexpr u32 kMaxLocal = 13;   // qubits resident in LDS
constexpr u32 kLowFixed = 3;    // qubits 0..2 are local in every stage: a tile is made of 128-byte runs
constexpr u32 kMinQubits = 4;   // smaller circuits run on 4 qubits (extra qubits stay |0>)

// Sub-operation kinds (low 4 bits of DSub::type).
// LAYER: CZ gates, then one 2x2 matrix on each block bit of a mask.  type bits
//   8..11: the block-bit mask; bits 4..7: those whose matrix is two shears; bits 16..31: the sign pattern over the register
//   block of the CZs between two block bits; bit 15: a and m hold, for block
//   bit i, the mask of local positions outside the block that share a CZ with
//   it (16 bits each: a = M0 | M1 << 16, m = M2 | M3 << 16), so the sign of
//   register slot j changes with the parity of base & M_i where bit i of j is
//   set; bits 12..14: the number (<= 4) of CZs between two positions outside
//   the block, byte c of pairs = p | q << 4; nx: the number (<= 8) of CZs between a
//   local position and a qubit outside the window, item c of x (16 bits each) =
//   tile bit | p << 8, p the local position or 0x80 | block bit.
//   data: the matrices (4 complex each; a, b and two unused for shears) of the mask's bits
//   in ascending order.
// D2: 4x4 on block bits byte 0 / byte 1 of a; DK: 2^K x 2^K on the block;
// DIAG: diagonal on the m qubits in the bytes of a (a local position, or kTileQubit
// | tile bit for a qubit outside the window).
// ZROT: amplitudes with even parity of the index bits of a mask times c + i s, the others
// times c - i s; a = mask of local positions outside the block | block-bit mask << 16, x[0]:
// mask of tile bits, data: c + i s.
// DEPOL (density matrices, column bits c and row bits r of m qubits): entries whose row and
// column bits differ times s; those where they agree times s plus t times their sum; a = block bits
// c0, r0, c1, r1 in bytes, m: qubits (1 or 2), data: s + i t.
enum : u32 { SUB_LAYER = 0, SUB_D2 = 1, SUB_DK = 2, SUB_DIAG = 3, SUB_ZROT = 4, SUB_DEPOL = 5 };
// bits 16 i .. 16 i + 15: the register-block indices j (< 16) with bit i set
constexpr u64 kBlockPatterns = 0xFF00F0F0CCCCAAAAull;
constexpr u32 kCzPairsMax = 4;
constexpr u32 kCzTileMax = 8;
constexpr u32 kTileQubit = 0x40;  // in a stage's operations: qubit kTileQubit | i is tile bit i

// Qubit lists are packed one byte per entry into 64-bit words so that the
// kernel indexes them with shifts (a runtime index into an array would put it
// in private memory).
struct DStage {
    u64 win[2];   // local bit kLowFixed + i <-> qubit byte i of win (i < lq - kLowFixed <= 10)
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
    u32 pool0;                // first pool entry of the pass
    // set in the first pass of a chunk of passes: bytes of the chunk's sub-operations, and of its
    // pool entries << 16, for warm_program
    u32 warm;
};
constexpr u32 kWarmBytes = 6144;  // per chunk: the scalar cache holds 16 KiB for two CUs
constexpr u32 kPassHasDiag = 1;
struct DSub {
    u32 type;
    u32 a;      // D2: block-bit indices (bytes); DIAG: local positions (bytes); LAYER: CZ masks
    u32 m;      // DIAG: qubit count; LAYER: CZ masks
    u32 data;   // offset into the complex pool
    u32 pairs;  // LAYER: CZs between two positions outside the block
    u32 grad0;  // LAYER: position in Flat::grads of the first matrix in gmask
    u32 gmask;  // LAYER: block bits whose matrix belongs to an operation with grad set
    u32 nx;     // LAYER: CZs with a qubit outside the window
    u64 x[2];
};
struct DTerm {
    u64 bf, pf;
    u32 rot, pad;
    double coef;
};

struct HOp {
    // 0 dense, 1 diag, 2 cz, 3 exp(i phi Z...Z) on q with m[0] = exp(i phi),
    // 4 depol on q = c0, r0 (, c1, r1) with m[0] = s + i t
    u32 type;
    bool dense() const { return type == 0 || type == 4; }  // mixes amplitudes: needs its qubits in a block
    std::vector<u32> q;
    std::vector<cx> m;
    bool reduced = false;  // single-qubit dense: m = {a, b, 0, 0} for [[1, 0], [b, 1]] [[1, a], [0, 1]]
    long id = -1;       // the caller's number of a single-qubit dense operation (see Flat::mats)
    bool grad = false;  // listed in Flat::grads
    u64 mask() const {  // tile bits aside
        u64 r = 0;
        for (u32 x : q)
            if (x < kTileQubit) r |= 1ULL << x;
        return r;
    }
};
struct HCirc {
    u32 n = 0;  // as given
    u32 ne = 0; // as run (>= kMinQubits)
    std::vector<HOp> ops;
    std::vector<DTerm> terms;
    // operations join qubit t with t + ne / 2 (a density matrix): windows of such pairs are
    // candidates too
    bool paired = false;
};


__host__ __device__ __forceinline__ u32 fold3(u32 x) { return ((x >> 3) ^ (x >> 6) ^ (x >> 9) ^ (x >> 12)) & 7u; }
__host__ __device__ __forceinline__ u32 slot_of(u32 x) { return x ^ fold3(x); }

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

// (x, y) <- (m0 x + m1 y, m2 x + m3 y), complex, on two pairs, updated in place; the matrix
// entries are wave-uniform (scalar registers).  Written as one asm block so the results land in
// the registers of the inputs: the sub-operation loop then keeps the register block at
// fixed registers instead of copying it at every merge point.  The last reader of each input
// writes a result into it (x.re holds the x.re chain from its 4th op on), so three temporaries
// per pair suffice.  The two pairs are interleaved instruction by instruction: a dependent FMA
// follows its producer 8 instructions later, which keeps the FP64 pipeline busy with only
// two waves per SIMD.
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

// pair_update2, or with `shear` set x += m0 y, then y += m1 x on both pairs: 8 multiply-adds
// per pair instead of 16.  The (uniform) choice is a branch inside the asm block: as two
// blocks under an if, the compiler copies the whole register block at the merge (16 64-bit moves
// per bit at K = 3, which cost what the shears save).
__device__ __forceinline__ void pair_either2(double2& x0, double2& y0, double2& x1, double2& y1, const double2 m0,
                                             const double2 m1, const double2 m2, const double2 m3, const u32 shear) {
    double tb0, tc0, td0, tb1, tc1, td1;
    asm("s_cmp_lg_u32 %[shear], 0\n\t"
        "s_cbranch_scc1 .Lshear%=\n\t"
        "v_mul_f64 %[tb0], %[m0i], %[xr0]\n\t"
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
        "v_fma_f64 %[yi1], %[m3r], %[yi1], %[td1]\n\t"
        "s_branch .Ldone%=\n\t"
        ".Lshear%=:\n\t"
        "v_fma_f64 %[xr0], %[m0r], %[yr0], %[xr0]\n\t"
        "v_fma_f64 %[xr1], %[m0r], %[yr1], %[xr1]\n\t"
        "v_fma_f64 %[xi0], %[m0r], %[yi0], %[xi0]\n\t"
        "v_fma_f64 %[xi1], %[m0r], %[yi1], %[xi1]\n\t"
        "v_fma_f64 %[xr0], -%[m0i], %[yi0], %[xr0]\n\t"
        "v_fma_f64 %[xr1], -%[m0i], %[yi1], %[xr1]\n\t"
        "v_fma_f64 %[xi0], %[m0i], %[yr0], %[xi0]\n\t"
        "v_fma_f64 %[xi1], %[m0i], %[yr1], %[xi1]\n\t"
        "v_fma_f64 %[yr0], %[m1r], %[xr0], %[yr0]\n\t"
        "v_fma_f64 %[yr1], %[m1r], %[xr1], %[yr1]\n\t"
        "v_fma_f64 %[yi0], %[m1r], %[xi0], %[yi0]\n\t"
        "v_fma_f64 %[yi1], %[m1r], %[xi1], %[yi1]\n\t"
        "v_fma_f64 %[yr0], -%[m1i], %[xi0], %[yr0]\n\t"
        "v_fma_f64 %[yr1], -%[m1i], %[xi1], %[yr1]\n\t"
        "v_fma_f64 %[yi0], %[m1i], %[xr0], %[yi0]\n\t"
        "v_fma_f64 %[yi1], %[m1i], %[xr1], %[yi1]\n\t"
        ".Ldone%=:"
        : [xr0] "+v"(x0.x), [xi0] "+v"(x0.y), [yr0] "+v"(y0.x), [yi0] "+v"(y0.y), [xr1] "+v"(x1.x),
          [xi1] "+v"(x1.y), [yr1] "+v"(y1.x), [yi1] "+v"(y1.y), [tb0] "=&v"(tb0), [tc0] "=&v"(tc0),
          [td0] "=&v"(td0), [tb1] "=&v"(tb1), [tc1] "=&v"(tc1), [td1] "=&v"(td1)
        : [m0r] "s"(m0.x), [m0i] "s"(m0.y), [m1r] "s"(m1.x), [m1i] "s"(m1.y), [m2r] "s"(m2.x), [m2i] "s"(m2.y),
          [m3r] "s"(m3.x), [m3i] "s"(m3.y), [shear] "s"(shear)
        : "scc");
}

// v <- v (c + i s) on two amplitudes, complex, in place; c uniform, s per lane.
__device__ __forceinline__ void phase2(double2& v, double2& w, const double c, const double sv, const double sw) {
    double t0, u0, t1, u1;
    asm("v_mul_f64 %[t0], %[sv], %[vi]\n\t"
        "v_mul_f64 %[t1], %[sw], %[wi]\n\t"
        "v_mul_f64 %[u0], %[sv], %[vr]\n\t"
        "v_mul_f64 %[u1], %[sw], %[wr]\n\t"
        "v_fma_f64 %[vr], %[c], %[vr], -%[t0]\n\t"
        "v_fma_f64 %[wr], %[c], %[wr], -%[t1]\n\t"
        "v_fma_f64 %[vi], %[c], %[vi], %[u0]\n\t"
        "v_fma_f64 %[wi], %[c], %[wi], %[u1]"
        : [vr] "+v"(v.x), [vi] "+v"(v.y), [wr] "+v"(w.x), [wi] "+v"(w.y), [t0] "=&v"(t0), [t1] "=&v"(t1),
          [u0] "=&v"(u0), [u1] "=&v"(u1)
        : [c] "s"(c), [sv] "v"(sv), [sw] "v"(sw));
}
// exp(i phi Z...Z) on a register block: slot j gets c + i s or c - i s by the parity of its
// block bits in bm (uniform) and the sign that s already carries.
template <int K>
__device__ __forceinline__ void zrot_block(double2 (&v)[1 << K], u32 bm, const double c, const double s) {
    u32 pat = 0;  // bit j: odd parity of j & bm
#pragma unroll
    for (int b = 0; b < K; ++b) pat ^= (0u - ((bm >> b) & 1u)) & (u32)((kBlockPatterns >> (16 * b)) & 0xffffu);
    const int hi = __double2hiint(s), lo = __double2loint(s);
#pragma unroll
    for (int j = 0; j < (1 << K); j += 2)
        phase2(v[j], v[j + 1], c, __hiloint2double(hi ^ (int)((pat << (31 - j)) & 0x80000000u), lo),
               __hiloint2double(hi ^ (int)((pat << (30 - j)) & 0x80000000u), lo));
}


// One 2x2 matrix on block bit P of each of the G register blocks of a thread.
// With two blocks, the pair updates interleave pair q of block 0 with pair q of
// block 1; with one block, pairs q and q + 1.
// REDUCE: bit P of `reduced` marks a matrix given as two shears.
template <int K, int P, int G, bool REDUCE>
__device__ __forceinline__ void sub_d1(double2 (&v)[G][1 << K], const double2* mp, u32 reduced) {
    const double2 m0 = mp[0], m1 = mp[1], m2 = mp[2], m3 = mp[3];
    // the 2^(K-1) pairs (j, j | 2^P)
    constexpr int NP = 1 << (K - 1);
    auto pair_j = [](int q) { return ((q >> P) << (P + 1)) | (q & ((1 << P) - 1)); };
    auto update = [&](double2& x0, double2& y0, double2& x1, double2& y1) {
        if constexpr (REDUCE) pair_either2(x0, y0, x1, y1, m0, m1, m2, m3, reduced & (1u << P));
        else pair_update2(x0, y0, x1, y1, m0, m1, m2, m3);
    };
    if constexpr (G == 2) {
#pragma unroll
        for (int q = 0; q < NP; ++q)
            update(v[0][pair_j(q)], v[0][pair_j(q) | (1 << P)], v[1][pair_j(q)], v[1][pair_j(q) | (1 << P)]);
    } else {
#pragma unroll
        for (int q = 0; q < NP; q += 2)
            update(v[0][pair_j(q)], v[0][pair_j(q) | (1 << P)], v[0][pair_j(q + 1)], v[0][pair_j(q + 1) | (1 << P)]);
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

// DEPOL on block bits (C0, R0), and (C1, R1) unless C1 < 0: 2.5 operations per component for two
// qubits, where the 16 x 16 superoperator takes 64.
template <int K, int C0, int R0, int C1, int R1>
__device__ __forceinline__ void depol_block(double2 (&v)[1 << K], const double s, const double t) {
    auto bit = [](int j, int b) { return (j >> b) & 1; };
#pragma unroll
    for (int j = 0; j < (1 << K); ++j) {
        // j: the member of its set of agreeing entries with all column bits 0
        if (bit(j, C0) || bit(j, R0)) continue;
        if (C1 >= 0 && (bit(j, C1 < 0 ? 0 : C1) || bit(j, R1 < 0 ? 0 : R1))) continue;
        const int d0 = (1 << C0) | (1 << R0), d1 = C1 >= 0 ? (1 << (C1 < 0 ? 0 : C1)) | (1 << (R1 < 0 ? 0 : R1)) : 0;
        double2 sum = cadd(v[j], v[j | d0]);
        if (C1 >= 0) sum = cadd(sum, cadd(v[j | d1], v[j | d0 | d1]));
        const double2 add = cscale(sum, t);
#pragma unroll
        for (int i = 0; i < (1 << K); ++i) {
            // the entries of j's group: all settings of the operation's bits
            if ((i & ~(d0 | d1)) != (j & ~(d0 | d1))) continue;
            const bool agree = bit(i, C0) == bit(i, R0) && (C1 < 0 || bit(i, C1 < 0 ? 0 : C1) == bit(i, R1 < 0 ? 0 : R1));
            v[i] = agree ? make_double2(fma(v[i].x, s, add.x), fma(v[i].y, s, add.y)) : cscale(v[i], s);
        }
    }
}
#define QM_DEPOL1_CASE(A, B)                 \
    case (A) * 4 + (B):                      \
        depol_block<4, A, B, -1, -1>(v, s, t); \
        break;
#define QM_DEPOL2_CASE(A, B, C, D)         \
    case (A) * 4 + (B):                    \
        depol_block<4, A, B, C, D>(v, s, t); \
        break;
__device__ __forceinline__ void apply_depol(double2 (&v)[16], u32 a, u32 m, const double s, const double t) {
    // the pair (c, r) is symmetric, and with two qubits the second pair is what is left of the block
    const u32 c = byte_at(a, 0), r = byte_at(a, 1), lo = min(c, r), hi = max(c, r);
    if (m == 1) {
        switch (lo * 4 + hi) {
            QM_DEPOL1_CASE(0, 1) QM_DEPOL1_CASE(0, 2) QM_DEPOL1_CASE(0, 3) QM_DEPOL1_CASE(1, 2) QM_DEPOL1_CASE(1, 3)
            QM_DEPOL1_CASE(2, 3)
            default: break;
        }
    } else {
        switch (lo * 4 + hi) {
            QM_DEPOL2_CASE(0, 1, 2, 3) QM_DEPOL2_CASE(0, 2, 1, 3) QM_DEPOL2_CASE(0, 3, 1, 2) QM_DEPOL2_CASE(1, 2, 0, 3)
            QM_DEPOL2_CASE(1, 3, 0, 2) QM_DEPOL2_CASE(2, 3, 0, 1)
            default: break;
        }
    }
}
#undef QM_DEPOL1_CASE
#undef QM_DEPOL2_CASE

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

// hi_tab[j] = global offset of local index j << kLowFixed (the window qubits kLowFixed.. of the
// stage).  TI = u32 holds offsets below 2^32 (states of at most 32 qubits);
// larger states use u64.
template <typename TI>
__device__ __forceinline__ void build_hi_tab(TI* hi_tab, u32 lq, const DStage& sg) {
    const u64 win0 = sg.win[0], win1 = sg.win[1];
    for (u32 j = threadIdx.x; j < (1u << (lq - kLowFixed)); j += blockDim.x) {
        TI o = 0;
        for (u32 i = 0; i + kLowFixed < lq; ++i) o |= (TI)((j >> i) & 1u) << byte_at(i < 8 ? win0 : win1, i & 7);
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

template <typename TI>
__device__ __forceinline__ u64 tile_index(u64 tb, const TI* hi_tab, u32 i) {
    return tb + hi_tab[i >> kLowFixed] + (i & ((1u << kLowFixed) - 1));
}

// The signs that the CZ gates of a LAYER give a register block with block base
// `base` (local index with zeros at the block positions): bit j of the result set
// means that amplitude j changes sign.  base is zero at the block positions, so a
// local position p outside the block is (base >> p) & 1 for the whole block.
// A qubit outside the window is a bit of the tile index: those CZs turn into uniform bits
// (block positions) or into one more mask of local positions (scalar work).
template <int K>
__device__ __forceinline__ u32 layer_signs(const DSub& sub, u32 base, u64 tile) {
    u32 sgn = sub.type >> 16;
    if (sub.nx) {
        u32 mask = 0;
        for (u32 c = 0; c < sub.nx; ++c) {
            const u32 w = (u32)((c < 4 ? sub.x[0] : sub.x[1]) >> (16 * (c & 3u))) & 0xffffu, p = w >> 8;
            const u32 on = (u32)(tile >> (w & 63u)) & 1u;
            if (p & 0x80u) sgn ^= (0u - on) & (u32)(kBlockPatterns >> (16 * (p & 3u))) & 0xffffu;
            else mask ^= on << p;
        }
        sgn ^= 0u - ((u32)__popc(base & mask) & 1u);
    }
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
// block base base[g].  The sub-operation is decoded once for all blocks.  REDUCE = false: no
// reduced matrices occur.
template <int K, int G, bool REDUCE = true>
__device__ __forceinline__ void apply_layer(double2 (&v)[G][1 << K], const DSub& sub, const u32 (&base)[G],
                                            const double2* __restrict__ pool, u64 tile) {
    const u32 d1 = (sub.type >> 8) & 15u;
    if ((sub.type >> 12) | sub.nx) {
        u32 sgn[G];
#pragma unroll
        for (int g = 0; g < G; ++g) sgn[g] = layer_signs<K>(sub, base[g], tile);
#pragma unroll
        for (int g = 0; g < G; ++g) flip_signs<K>(v[g], sgn[g]);
    }
    const double2* mp = pool + sub.data;
    const u32 red = (sub.type >> 4) & 15u;
    if (d1 & 1u) {
        sub_d1<K, 0, G, REDUCE>(v, mp, red);
        mp += 4;
    }
    if (d1 & 2u) {
        sub_d1<K, 1, G, REDUCE>(v, mp, red);
        mp += 4;
    }
    if constexpr (K > 2)
        if (d1 & 4u) {
            sub_d1<K, 2, G, REDUCE>(v, mp, red);
            mp += 4;
        }
    if constexpr (K > 3)
        if (d1 & 8u) sub_d1<K, 3, G, REDUCE>(v, mp, red);
}

// The sub-operations of one pass on the G register blocks of groups gi0,
// gi0 + T, ..., read from and written back to LDS.  slot_of is linear over
// GF(2), so the slot of base | off[j] is slot_of(base) ^ (XOR of sbit[i] over
// the bits i of j): each lane forms its 2^K slots from the K per-bit offsets
// (the empty asm keeps every partial XOR in a vector register, so the compiler
// does not form the 2^K uniform combinations in scalar registers, which spill).
// WIDE = false: only LAYER (with full matrices) and D2 sub-operations occur.
template <int K, u32 T, int G, bool WIDE = true>
__device__ __forceinline__ void pass_groups(double2* st, const DPass& ps, const u32 (&sbit)[K], u32 gi0,
                                            const DSub* __restrict__ subs, const double2* __restrict__ pool,
                                            u64 tile) {
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
        static_assert(SUB_LAYER == 0 && SUB_ZROT == 4, "the test below");
        while ((sub.type & 11u) == 0) {
            // a chain of conditional in-place updates (a ZROT has none of LAYER's parts)
            if (WIDE && (sub.type & 4u)) {
                const double2 z = pool[sub.data];
                const u32 odd = (u32)__popcll(tile & sub.x[0]);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int f = (int)((odd + (u32)__popc(base[g] & sub.a & 0xffffu)) << 31);
                    zrot_block<K>(v[g], sub.a >> 16, z.x, __hiloint2double(__double2hiint(z.y) ^ f, __double2loint(z.y)));
                }
            }
            apply_layer<K, G, WIDE>(v, sub, base, pool, tile);
            if (++k == ps.nsub) break;
            sub = subs[ps.sub0 + k];
        }
        if (k == ps.nsub) break;
        const u32 kind = sub.type & 15u;
        const double2* mp = pool + sub.data;
        if constexpr (WIDE && K == 4) {
            if (kind == SUB_DEPOL) {
                const double2 f = mp[0];
#pragma unroll
                for (int g = 0; g < G; ++g) apply_depol(v[g], sub.a, sub.m, f.x, f.y);
                ++k;
                continue;
            }
        }
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
            // base or, for a block position, bit j of the block pattern; or a tile bit
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
                for (int i = 0; i < 4; ++i) {
                    const u32 p = byte_at(sub.a, i);
                    const u32 bit = p & kTileQubit ? (u32)(tile >> (p & 63u)) & 1u : (base[g] >> (p & 31u)) & 1u;
                    tbit[i] = i < (int)sub.m ? bit : 0u;
                }
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

// Brings a chunk of the program into the scalar cache: every wave reads its share of the cache
// lines, all at once.  Read on demand, each line is a miss of several hundred cycles in a chain
// (descriptor, then matrix) that nothing hides when a CU runs a single tile: a 20-qubit
// circuit of 10 brickwork layers (256 tiles for 256 CUs) takes 127 us instead of 166.
// (Plain indexed reads: turning the pointer into an integer would let the compiler assume that
// stores change the program, and read it with vector loads.)
__device__ __forceinline__ void warm_lines(const u32* __restrict__ p, u32 bytes) {
    const u32 n = (bytes + 63) / 64;  // steps of a line, and the last word
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    for (u32 i = wave; i <= n && bytes; i += 4 * nw) {
        u32 x[4];
#pragma unroll
        for (u32 k = 0; k < 4; ++k) x[k] = p[min((i + k * nw) * 16, bytes / 4 - 1)];
        asm volatile("" ::"s"(x[0]), "s"(x[1]), "s"(x[2]), "s"(x[3]));
    }
}
__device__ __forceinline__ void warm_program(const DPass& ps, const DSub* __restrict__ subs,
                                             const double2* __restrict__ pool) {
    warm_lines(reinterpret_cast<const u32*>(subs + ps.sub0), ps.warm & 0xffffu);
    warm_lines(reinterpret_cast<const u32*>(pool + ps.pool0), ps.warm >> 16);
}

// Applies passes [pass0, pass0 + npass) to the 2^lq amplitudes in LDS with a
// work-group of T threads (of at most T if it has fewer groups than T), `tile`: the
// tile's index; ends with a barrier after every pass.  With G = 2
// and exactly 2 T groups of 2^K amplitudes, every thread holds two register
// blocks and decodes each sub-operation once for both.
template <int K, u32 T, int G, bool WIDE = true>
__device__ __forceinline__ void run_passes(double2* st, u32 lq, const DPass* __restrict__ passes, u32 pass0,
                                           u32 npass, const DSub* __restrict__ subs,
                                           const double2* __restrict__ pool, u64 tile) {
    constexpr int D = 1 << K;
    const u32 ngroups = (1u << lq) >> K;
    for (u32 p = 0; p < npass; ++p) {
        const DPass ps = passes[pass0 + p];
        if (p > 0 && ps.warm) warm_program(ps, subs, pool);  // the first chunk: see the callers
        u32 sbit[K];
#pragma unroll
        for (int i = 0; i < K; ++i) sbit[i] = ps.sbit[i];
        if (G == 2 && ngroups == 2 * T && !(ps.flags & kPassHasDiag)) {
            pass_groups<K, T, G, WIDE>(st, ps, sbit, threadIdx.x, subs, pool, tile);
        } else if (ngroups == T) {
            pass_groups<K, T, 1, WIDE>(st, ps, sbit, threadIdx.x, subs, pool, tile);
        } else {
            for (u32 g = threadIdx.x; g < ngroups; g += blockDim.x)
                pass_groups<K, T, 1, WIDE>(st, ps, sbit, g, subs, pool, tile);
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ host side
void mat_mul(const std::vector<cx>& a, const std::vector<cx>& b, std::vector<cx>& out, int d) {
    out.assign((size_t)d * d, 0.0);
    for (int i = 0; i < d; ++i)
        for (int k = 0; k < d; ++k)
            for (int j = 0; j < d; ++j) out[i * d + j] += mul(a[i * d + k], b[k * d + j]);
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

u32 pool_put(Flat& f, const std::vector<cx>& m) {
    const u32 off = (u32)f.pool.size();
    for (const cx& z : m) f.pool.push_back(make_double2((double)z.real(), (double)z.imag()));
    return off;
}

// The window (or block) of the next stage (or pass).  Operations are scanned in order; a
// dense operation is taken if its qubits lie in the window, a diagonal one if it touches
// the window at all (a qubit outside is a constant there); a dense operation that is not
// taken blocks its qubits for everything after it.  Diagonal operations that do not touch the
// window block nothing: they commute with what is taken.  Candidates: the window that grows
// in scan order (any circuit), and every run of adjacent qubits (chains and grids, where the
// order of the gate list would spread the window over the register and leave each stage a few
// layers: 26-qubit brickwork, 20 layers, 12-qubit windows: 9 stages, 26 in list
// order with 13; 20-qubit ansatz backward: 24 -> 8).
// The one with the most dense work wins.
struct Picker {
    struct Item {
        u64 mask;
        u32 weight;  // 0: diagonal
        bool grad;
    };
    std::vector<Item> items;
    std::vector<u32> rest;  // what is left, in order
    u64 left = 0;           // its dense work

    static u32 weight_of(const HOp& o) { return o.type == 0 ? 1u << (o.q.size() - 1) : o.type == 4 ? 1u : 0u; }
    void add(const HOp& o) {
        rest.push_back((u32)items.size());
        items.push_back({o.mask(), weight_of(o), o.grad});
        left += items.back().weight;
    }
    // Scans with window w (grown up to `most` qubits if `grow`); returns the dense work taken.
    u64 scan(u64& w, bool grow, u32 most, size_t max_grads, std::vector<u32>* sel) const {
        u64 blocked = 0, work = 0;
        size_t grads = 0;
        for (u32 i : rest) {
            const Item& it = items[i];
            if (it.mask & blocked) {
                // (a diagonal one that a fixed window does not touch orders nothing in it)
                if (it.weight || grow || (it.mask & w)) blocked |= it.mask;
                if ((blocked & w) == w && (!grow || (u32)__builtin_popcountll(w) >= most)) break;
                continue;
            }
            if (it.weight == 0) {
                if (sel) sel->push_back(i);
                continue;
            }
            const u64 m = it.mask | w;
            const bool fits = m == w || (grow && (u32)__builtin_popcountll(m) <= most);
            if (fits && (!it.grad || grads < max_grads)) {
                w = m;
                work += it.weight;
                grads += it.grad ? 1 : 0;
                if (sel) sel->push_back(i);
            } else {
                blocked |= it.mask;
                if ((blocked & w) == w && (!grow || (u32)__builtin_popcountll(w) >= most)) break;
            }
        }
        return work;
    }
    // Picks a window of at most `most` positions out of [0, n) that contains `fixed`, and
    // what it takes; the window is filled up to min(n, most) positions.
    // `paired`: also windows of qubits s, s + 1, ... of [0, n / 2) with their partners n / 2 above.
    u64 pick(u32 n, u64 fixed, u32 low, u32 most, size_t max_grads, std::vector<u32>& sel, bool paired = false) {
        u64 best = fixed;
        u64 work = scan(best, true, most, max_grads, nullptr);
        const u32 f = most - low;
        bool grow = true;
        // (a window that takes all there is cannot be beaten)
        for (u32 s = low; s + f <= n && work < left; ++s) {
            u64 w = fixed | (((1ULL << f) - 1) << s);
            const u64 c = scan(w, false, most, max_grads, nullptr);
            if (c > work) {
                work = c;
                best = w;
                grow = false;
            }
        }
        for (u32 s = 0; paired && s < n / 2 && work < left; ++s) {
            u64 w = fixed;
            for (u32 q = s; q < n / 2; ++q) {
                const u64 m = w | (1ULL << q) | (1ULL << (q + n / 2));
                if ((u32)__builtin_popcountll(m) > most) break;
                w = m;
            }
            const u64 c = scan(w, false, most, max_grads, nullptr);
            if (c > work) {
                work = c;
                best = w;
                grow = false;
            }
        }
        u64 w = grow ? fixed : best;
        sel.clear();
        scan(w, grow, most, max_grads, &sel);
        // fill the window: with the qubits of diagonal operations that wait, then the lowest
        auto room = [&] { return (u32)__builtin_popcountll(w) < std::min(n, most); };
        for (u32 i : sel)
            for (u64 m = items[i].mask & ~w; m && room(); m &= m - 1) w |= m & (~m + 1);
        for (u32 q = 0; q < n && room(); ++q) w |= 1ULL << q;
        // a diagonal operation outside the window stays for a later one
        sel.erase(std::remove_if(sel.begin(), sel.end(), [&](u32 i) { return !(items[i].mask & w); }), sel.end());
        return w;
    }
    void take(const std::vector<u32>& sel) {  // sel is ascending in `rest` order
        size_t k = 0, out = 0;
        for (size_t i = 0; i < rest.size(); ++i) {
            if (k < sel.size() && rest[i] == sel[k]) {
                left -= items[rest[i]].weight;
                ++k;
            } else {
                rest[out++] = rest[i];
            }
        }
        rest.resize(out);
    }
};

// Passes of one stage: ops (already in local positions) -> DPass/DSub.
void schedule_passes(Flat& f, const std::vector<HOp>& ops, u32 lq, u32 K, DStage& sg) {
    sg.pass0 = (u32)f.passes.size();
    sg.npass = 0;
    Picker pk;
    size_t dense_left = 0;
    for (const HOp& o : ops) {
        pk.add(o);
        dense_left += o.dense();
    }
    std::vector<u32> sel;
    while (!pk.rest.empty()) {
        const u64 block = pk.pick(lq, 0, 0, K, ~size_t(0), sel);
        for (u32 i : sel) dense_left -= ops[i].dense();
        if (dense_left == 0) sel = pk.rest;  // the last pass takes every diagonal operation that is left
        pk.take(sel);
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
        ps.pool0 = (u32)f.pool.size();
        auto bit_of = [&](u32 p) -> u32 {
            for (u32 i = 0; i < K; ++i)
                if (bpos[i] == p) return i;
            return 0;
        };
        // Levels: an operation goes to the first level after what it does not commute
        // with (only block bits carry dense operations); a level is its diagonal
        // operations, then its matrices on distinct block bits.
        std::vector<std::vector<u32>> levels;
        {
            u32 dense_at[4] = {0, 0, 0, 0}, diag_at[4] = {0, 0, 0, 0};
            for (u32 i : sel) {
                const HOp& o = ops[i];
                u32 lv = 1;
                for (u32 q : o.q) {
                    if (q >= kTileQubit || !((block >> q) & 1)) continue;
                    const u32 b = bit_of(q);
                    lv = std::max(lv, dense_at[b] + 1);
                    if (o.dense()) lv = std::max(lv, diag_at[b]);
                }
                for (u32 q : o.q) {
                    if (q >= kTileQubit || !((block >> q) & 1)) continue;
                    u32& at = (o.dense() ? dense_at : diag_at)[bit_of(q)];
                    at = std::max(at, lv);
                }
                if (levels.size() < lv) levels.resize(lv);
                levels[lv - 1].push_back(i);
            }
        }
        std::vector<const HOp*> pend_d1(K, nullptr);
        u32 d1mask = 0, redmask = 0, cz_const = 0, npair = 0, pairs = 0, nx = 0;
        u64 xs[2] = {0, 0};
        u32 czmask[4] = {0, 0, 0, 0};
        bool cz_any = false;
        auto flush = [&]() {
            if (d1mask == 0 && !cz_any) return;
            DSub sb{};
            const bool masks = (czmask[0] | czmask[1] | czmask[2] | czmask[3]) != 0;
            sb.type = SUB_LAYER | (redmask << 4) | (d1mask << 8) | (npair << 12) | (masks ? 0x8000u : 0u) | (cz_const << 16);
            sb.a = czmask[0] | (czmask[1] << 16);
            sb.m = czmask[2] | (czmask[3] << 16);
            sb.pairs = pairs;
            sb.nx = nx;
            sb.x[0] = xs[0];
            sb.x[1] = xs[1];
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
            d1mask = redmask = 0;
            cz_const = 0;
            npair = 0;
            pairs = 0;
            nx = 0;
            xs[0] = xs[1] = 0;
            std::fill(czmask, czmask + 4, 0u);
            cz_any = false;
        };
        const u32 jmask = (1u << (1u << K)) - 1;
        auto add_cz = [&](u32 p0, u32 p1) {
            if (p0 >= kTileQubit) std::swap(p0, p1);
            if (p1 >= kTileQubit) {
                if (nx == kCzTileMax) flush();
                const u32 in = ((block >> p0) & 1) ? 0x80u | bit_of(p0) : p0;
                xs[nx >> 2] |= (u64)((p1 & 63u) | (in << 8)) << (16 * (nx & 3));
                ++nx;
                cz_any = true;
                return;
            }
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
        for (const auto& level : levels) {
            for (u32 i : level) {
                const HOp& o = ops[i];
                if (o.type != 1) continue;
                DSub sb{};
                ps.flags |= kPassHasDiag;
                sb.type = SUB_DIAG;
                sb.m = (u32)o.q.size();
                for (size_t k = 0; k < o.q.size(); ++k) sb.a |= o.q[k] << (8 * k);
                sb.data = pool_put(f, o.m);
                f.subs.push_back(sb);
            }
            for (u32 i : level) {
                const HOp& o = ops[i];
                if (o.type != 3) continue;
                DSub sb{};
                sb.type = SUB_ZROT;
                for (u32 q : o.q) {
                    if (q >= kTileQubit) sb.x[0] |= 1ULL << (q & 63u);
                    else if ((block >> q) & 1) sb.a |= 0x10000u << bit_of(q);
                    else sb.a |= 1u << q;
                }
                sb.data = pool_put(f, o.m);
                f.subs.push_back(sb);
            }
            for (u32 i : level)
                if (ops[i].type == 2) add_cz(ops[i].q[0], ops[i].q[1]);
            for (u32 i : level) {
                const HOp& o = ops[i];
                if (o.type != 0 || o.q.size() != 1) continue;
                pend_d1[bit_of(o.q[0])] = &o;
                d1mask |= 1u << bit_of(o.q[0]);
                if (o.reduced) redmask |= 1u << bit_of(o.q[0]);
            }
            flush();
            for (u32 i : level) {
                const HOp& o = ops[i];
                if (!o.dense() || o.q.size() == 1) continue;
                DSub sb{};
                if (o.type == 4) {
                    sb.type = SUB_DEPOL;
                    sb.m = (u32)o.q.size() / 2;
                    for (size_t k = 0; k < o.q.size(); ++k) sb.a |= bit_of(o.q[k]) << (8 * k);
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
                    std::vector<cx> M((size_t)D * D, 0.0);
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
        }
        ps.nsub = (u32)f.subs.size() - ps.sub0;
        f.passes.push_back(ps);
        ++sg.npass;
    }
    // chunks of passes for warm_program
    for (u32 p = sg.pass0; p < sg.pass0 + sg.npass;) {
        auto end_of = [&](u32 q, bool pool) {
            const bool last = q + 1 == f.passes.size();
            return pool ? (last ? (u32)f.pool.size() : f.passes[q + 1].pool0)
                        : (last ? (u32)f.subs.size() : f.passes[q + 1].sub0);
        };
        DPass& head = f.passes[p];
        u32 q = p;
        for (;; ++q) {
            const u32 bs = (end_of(q, false) - head.sub0) * (u32)sizeof(DSub);
            const u32 bp = (end_of(q, true) - head.pool0) * (u32)sizeof(double2);
            if (q > p && bs + bp > kWarmBytes) break;
            head.warm = std::min(bs, 2 * kWarmBytes) | std::min(bp, 2 * kWarmBytes) << 16;
            if (q + 1 == sg.pass0 + sg.npass) {
                ++q;
                break;
            }
        }
        p = q;
    }
}

// Stages (windows of lq_cap qubits including those below `low_fixed`) for circuits above
// lq_cap qubits; a single identity stage otherwise.  A stage takes at most `max_grads`
// operations with grad set.  Returns the number of stages appended.
u32 schedule_circuit(Flat& f, const HCirc& c, u32 K, u32 lq_cap = kMaxLocal, size_t max_grads = ~size_t(0)) {
    const u32 n = c.ne, lq = std::min(n, lq_cap);
    if (n <= lq_cap && max_grads == ~size_t(0)) {
        DStage sg{};
        for (u32 i = 0; i + kLowFixed < lq; ++i) set_byte(sg.win[i >> 3], i & 7, kLowFixed + i);
        schedule_passes(f, c.ops, lq, K, sg);
        f.stages.push_back(sg);
        return 1;
    }
    Picker pk;
    for (const HOp& o : c.ops) pk.add(o);
    const u64 low = (1ULL << kLowFixed) - 1;
    u32 count = 0;
    std::vector<u32> sel;
    do {  // a circuit without gates still needs one stage to initialise |0>
        const u64 win = pk.pick(n, low, kLowFixed, lq, max_grads, sel, c.paired);
        pk.take(sel);
        DStage sg{};
        u32 local_of[64];
        u32 wi = 0, ci = 0;
        for (u32 q = 0; q < n; ++q) {
            if (q < kLowFixed) {
                local_of[q] = q;
            } else if ((win >> q) & 1) {
                local_of[q] = kLowFixed + wi;
                set_byte(sg.win[wi >> 3], wi & 7, q);
                ++wi;
            } else {
                local_of[q] = kTileQubit | ci;
                set_byte(sg.comp[ci >> 3], ci & 7, q);
                ++ci;
            }
        }
        std::vector<HOp> ops;
        ops.reserve(sel.size());
        for (u32 i : sel) {
            ops.push_back(c.ops[i]);
            for (u32& q : ops.back().q) q = local_of[q];
        }
        schedule_passes(f, ops, lq, K, sg);
        f.stages.push_back(sg);
        ++count;
    } while (!pk.rest.empty());
    return count;
}

// Gates in the C ABI form -> internal operations.
//   * Consecutive single-qubit gates on a qubit are multiplied together.
//   * Diagonal operations (CZ, ZROT, DIAG) commute, so a single-qubit diagonal waits in `pend`
//     and is multiplied into the next dense operation on its qubit, or, at the end, into
//     the last one.
//   * CNOT(c, t) = H_t CZ(c, t) H_t with H = [[1, 1], [1, -1]] before and half of it after
//     the CZ: both exact, where 1/sqrt(2) twice would change the norm by 1.4e-16 per CNOT.
//   * A diagonal gate with entries of modulus 1 is a product of exp(i phi Z...Z) over subsets of
//     its qubits: phases on single qubits wait as above, the others become ZROT when they
//     are few (a two-qubit gate has one), else the gate stays a DIAG.  Moduli that differ from 1
//     by more than rounding are kept (see diagonal).
struct Converter {
    HCirc& c;
    std::vector<long> last;        // last operation that touches each qubit
    std::vector<long> last_dense;  // last dense one
    struct Phase {
        cx d[2] = {1.0, 1.0};
        bool any = false;
    };
    std::vector<Phase> pend;

    explicit Converter(HCirc& circ) : c(circ), last(circ.ne, -1), last_dense(circ.ne, -1), pend(circ.ne) {}

    void push(HOp o) {
        c.ops.push_back(std::move(o));
        const long i = (long)c.ops.size() - 1;
        for (u32 q : c.ops.back().q) {
            last[q] = i;
            if (c.ops.back().dense()) last_dense[q] = i;
        }
    }
    void phase(u32 q, cx d0, cx d1) {
        pend[q].d[0] = mul(pend[q].d[0], d0);
        pend[q].d[1] = mul(pend[q].d[1], d1);
        pend[q].any = true;
    }
    void dense(const std::vector<u32>& q, std::vector<cx> m) {
        const u32 d = 1u << q.size();
        for (u32 t = 0; t < q.size(); ++t) {
            Phase& ph = pend[q[t]];
            if (!ph.any) continue;
            for (u32 r = 0; r < d; ++r)
                for (u32 col = 0; col < d; ++col) m[r * d + col] = mul(m[r * d + col], ph.d[(col >> t) & 1u]);
            ph = Phase{};
        }
        const long p = last[q[0]];
        if (p >= 0 && c.ops[p].type == 0 && c.ops[p].q == q && last[q.back()] == p && q.size() <= 2) {
            std::vector<cx> prod;
            mat_mul(m, c.ops[p].m, prod, (int)d);  // new after old
            c.ops[p].m = prod;
            return;
        }
        HOp o;
        o.type = 0;
        o.q = q;
        o.m = std::move(m);
        push(std::move(o));
    }
    void zrot(const std::vector<u32>& q, cx z) {
        if (q.size() == 1) {
            phase(q[0], z, std::conj(z));
            return;
        }
        HOp o;
        o.type = 3;
        o.q = q;
        o.m = {z};
        push(std::move(o));
    }
    void diagonal(const std::vector<u32>& q, const std::vector<cx>& m) {
        const u32 k = (u32)q.size(), d = 1u << k;
        if (k == 1) {
            phase(q[0], m[0], m[1]);
            return;
        }
        auto subset = [&](u32 s) {
            std::vector<u32> r;
            for (u32 t = 0; t < k; ++t)
                if ((s >> t) & 1) r.push_back(q[t]);
            return r;
        };
        for (u32 s = 1; s < d; ++s) {  // one exp(i phi Z...Z), entries as they are
            bool is = std::abs(std::abs(m[0]) - 1.0) < 1e-14;
            for (u32 i = 1; i < d && is; ++i) is = m[i] == ((__builtin_popcount(i & s) & 1) ? std::conj(m[0]) : m[0]);
            if (is) {
                zrot(subset(s), m[0]);
                return;
            }
        }
        bool unit = true;
        for (u32 i = 0; i < d && unit; ++i) unit = std::abs(std::norm(m[i]) - 1.0L) < 2e-14L;
        if (unit) {
            // log m_i = sum_s (-1)^popcount(i & s) (rho[s] + i phi[s]) / d.  What a double's rounding
            // leaves of the moduli (2^-53) may go; more of it is kept: rho of all and of single
            // qubits in the phases that wait, of more qubits by leaving the gate a DIAG.
            long double phi[16], rho[16];
            auto transform = [&](long double* x) {
                for (u32 h = 1; h < d; h <<= 1)
                    for (u32 i = 0; i < d; ++i)
                        if (!(i & h)) {
                            const long double a = x[i], b = x[i | h];
                            x[i] = a + b;
                            x[i | h] = a - b;
                        }
            };
            for (u32 i = 0; i < d; ++i) phi[i] = std::arg(m[i]);
            transform(phi);
            u32 many = 0;
            for (u32 s = 1; s < d; ++s) many += (s & (s - 1)) && std::abs(phi[s]) > 1e-15;
            bool kept = many <= 2;
            if (kept) {
                for (u32 i = 0; i < d; ++i) rho[i] = 0.5L * (std::norm(m[i]) - 1.0L);  // log |m_i| up to 1e-28
                transform(rho);
                for (u32 s = 0; s < d; ++s) {
                    if (std::abs(rho[s]) <= d * 0x1p-53L) rho[s] = 0.0L;
                    kept = kept && (rho[s] == 0.0L || !(s & (s - 1)));
                }
            }
            if (kept) {
                const cx g = std::polar(std::exp(rho[0] / d), phi[0] / d);
                phase(q[0], g, g);
                for (u32 s = 1; s < d; ++s) {
                    if (std::abs(phi[s]) <= 1e-15 && rho[s] == 0.0L) continue;
                    if (s & (s - 1)) zrot(subset(s), std::polar(1.0L, phi[s] / d));
                    else phase(q[__builtin_ctz(s)], std::polar(std::exp(rho[s] / d), phi[s] / d), std::polar(std::exp(-rho[s] / d), -phi[s] / d));
                }
                return;
            }
        }
        HOp o;
        o.type = 1;
        o.q = q;
        o.m = m;
        push(std::move(o));
    }
    void depol(const std::vector<u32>& q, cx st) {
        for (u32 x : q) flush(x);
        HOp o;
        o.type = 4;
        o.q = q;
        o.m = {st};
        push(std::move(o));
    }
    // What is left in pend: into the last dense operation on the qubit (only diagonal ones
    // follow it), else a diagonal operation of its own.
    void finish() {
        for (u32 q = 0; q < c.ne; ++q) flush(q);
    }
    void flush(u32 q) {
        {
            Phase& ph = pend[q];
            if (!ph.any) return;
            if (last_dense[q] >= 0 && c.ops[last_dense[q]].type == 0) {
                HOp& o = c.ops[last_dense[q]];
                const u32 d = 1u << o.q.size(), t = (u32)(std::find(o.q.begin(), o.q.end(), q) - o.q.begin());
                for (u32 r = 0; r < d; ++r)
                    for (u32 col = 0; col < d; ++col) o.m[r * d + col] = mul(o.m[r * d + col], ph.d[(r >> t) & 1u]);
            } else if (ph.d[0] != cx(1.0) || ph.d[1] != cx(1.0)) {
                HOp o;
                o.type = 1;
                o.q = {q};
                o.m = {ph.d[0], ph.d[1]};
                push(std::move(o));
            }
            ph = Phase{};
        }
    }
};

// A single-qubit unitary U = diag(p, q) [[1, 0], [b, 1]] [[1, a], [0, 1]] with p = u00,
// a = u01 / u00, q = det / u00, b = u10 / q, or X times that for X U where |u10| is the larger.  The
// monomial factor X^f diag passes what is diagonal (flipped on the qubit) and is multiplied into
// the next dense operation on the qubit, so all
// single-qubit matrices but the last on a qubit cost 8 multiply-adds per pair instead of 16 (the
// fused executors are bound by VALU issue: see qm_batch.hip).  A CZ passes as itself, a Z on the other
// qubit, which joins what waits there, and a sign if both are flipped; so X is taken only where every such
// qubit has a dense operation to come.  Without the flip a quarter of random
// matrices stayed whole: brickwork at 26 qubits 11.06 ms, with it 10.35.
// Scaling rows or columns by a diagonal changes no relative rounding error, and with
// the larger of two entries as p the shears add terms of at most sqrt(2) times the result's size, so
// the error is that of the full matrix.  Amplitudes are off by 1/p or 1/q until the diagonal is
// applied.  A matrix is left whole when |p| < 1/2, when that factor would exceed 2^200 in
// all, and when it is not unitary (or a multiple of a unitary).
void reduce_matrices(std::vector<HOp>& ops, u32 n) {
    // the next operation that mixes amplitudes on the qubit has a matrix to take the diagonal,
    // and so has every partner of a CZ up to there
    std::vector<bool> absorbed(ops.size(), false), flippable(ops.size(), false);
    {
        std::vector<bool> next(n, false), flip(n, false);
        for (size_t i = ops.size(); i-- > 0;) {
            const HOp& o = ops[i];
            if (o.type == 2) {
                const u32 x = o.q[0], y = o.q[1];
                flip[x] = flip[x] && next[y];
                flip[y] = flip[y] && next[x];
            }
            if (!o.dense()) continue;
            if (o.q.size() == 1) {
                absorbed[i] = next[o.q[0]];
                flippable[i] = flip[o.q[0]];
            }
            for (u32 q : o.q) next[q] = flip[q] = o.type == 0;
        }
    }
    struct Left {
        cx d[2] = {1.0, 1.0};
        bool any = false, flip = false;
        double bits = 0.0;  // |log2| of the larger factor that waits in d
    };
    std::vector<Left> left(n);
    double total = 0.0;
    for (size_t i = 0; i < ops.size(); ++i) {
        HOp& o = ops[i];
        u32 flips = 0;  // bits of the operation's index that stand for flipped qubits
        for (u32 t = 0; t < o.q.size(); ++t) flips |= (u32)left[o.q[t]].flip << t;
        if (o.type == 1 && flips) {
            std::vector<cx> m(o.m.size());
            for (u32 x = 0; x < m.size(); ++x) m[x] = o.m[x ^ flips];
            o.m = std::move(m);
        }
        if (o.type == 2 && flips) {
            for (u32 t = 0; t < 2; ++t)
                if ((flips >> t) & 1) {
                    Left& l = left[o.q[1 - t]];
                    l.d[1] = -l.d[1];
                    l.any = true;
                }
            if (flips == 3)
                for (cx& z : left[o.q[0]].d) z = -z;
        }
        if (o.type == 3 && (__builtin_popcount(flips) & 1)) o.m[0] = std::conj(o.m[0]);
        if (o.type != 0) continue;
        const u32 d = 1u << o.q.size();
        std::vector<cx> m(o.m);
        for (u32 t = 0; t < o.q.size(); ++t) {
            Left& l = left[o.q[t]];
            if (!l.any) continue;
            if (l.flip) {
                for (u32 r = 0; r < d; ++r)
                    for (u32 col = 0; col < d; ++col)
                        if (!((col >> t) & 1u)) std::swap(m[r * d + col], m[r * d + (col | (1u << t))]);
            }
            for (u32 r = 0; r < d; ++r)
                for (u32 col = 0; col < d; ++col) m[r * d + col] = mul(m[r * d + col], l.d[(col >> t) & 1u]);
        }
        bool shear = false, flip = false;
        if (absorbed[i]) {
            const cx* g = o.m.data();  // the operation itself: what waits may be no unitary
            const double c0 = std::norm(g[0]) + std::norm(g[2]), c1 = std::norm(g[1]) + std::norm(g[3]);
            const cx dot = mul(std::conj(g[0]), g[1]) + mul(std::conj(g[2]), g[3]);
            const u32 f = flips & 1u;  // the first column, once what waits has been multiplied in
            flip = flippable[i] && std::norm(g[2 + f]) > std::norm(g[f]);
            shear = c0 > 1e-6 && c0 < 1e6 && std::abs(c1 - c0) < 1e-12 * c0 && std::abs(dot) < 1e-12 * c0 &&
                    std::norm(g[(flip ? 2 : 0) + f]) >= 0.25 * c0;
        }
        o.m = std::move(m);
        for (u32 q : o.q) {
            total -= left[q].bits;
            left[q] = Left{};
        }
        if (!shear) continue;
        if (flip) {
            std::swap(o.m[0], o.m[2]);
            std::swap(o.m[1], o.m[3]);
        }
        const cx p = o.m[0], a = quot(o.m[1], o.m[0]), q = o.m[3] - mul(o.m[2], a);
        const double bits = std::max(std::abs(std::log2(std::abs(p))), std::abs(std::log2(std::abs(q))));
        if (!(total + bits < 200.0)) {
            if (flip) {
                std::swap(o.m[0], o.m[2]);
                std::swap(o.m[1], o.m[3]);
            }
            continue;
        }
        Left& l = left[o.q[0]];
        l.d[0] = p;
        l.d[1] = q;
        l.any = true;
        l.flip = flip;
        l.bits = bits;
        total += bits;
        o.m = {a, quot(o.m[2], q), 0.0, 0.0};
        o.reduced = true;
    }
}

// `density`: QM_BATCH_DEPOL is taken, and dense operations on t and t + n / 2 mark the circuit as
// paired.
bool convert_gates(u32 n, const qm_batch_gate* gates, UINT gate_count, HCirc& c, const char* what,
                   bool density = false) {
    c.n = n;
    c.ne = std::max<u32>(n, kMinQubits);
    Converter cv(c);
    for (UINT gi = 0; gi < gate_count; ++gi) {
        const qm_batch_gate& g = gates[gi];
        const u32 k = g.qubit_count;
        const bool two = g.kind == QM_BATCH_CZ || g.kind == QM_BATCH_CNOT;
        const bool depol = g.kind == QM_BATCH_DEPOL && density;
        if ((g.kind > QM_BATCH_CNOT && !depol) || k < 1 || k > 4 || (two && k != 2) || (depol && k != 2 && k != 4)) {
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
        if ((g.kind == QM_BATCH_DENSE || g.kind == QM_BATCH_DIAG || depol) && !g.matrix) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: gate %u: null matrix", what, gi);
            return false;
        }
        const std::vector<u32> q(g.qubits, g.qubits + k);
        const u32 d = 1u << k;
        std::vector<cx> m;
        if (two) {
            HOp cz;
            cz.type = 2;
            cz.q = q;
            if (g.kind == QM_BATCH_CNOT) cv.dense({q[1]}, {1.0, 1.0, 1.0, -1.0});
            cv.push(std::move(cz));
            if (g.kind == QM_BATCH_CNOT) cv.dense({q[1]}, {0.5, 0.5, 0.5, -0.5});
        } else if (depol) {
            cv.depol(q, cx(g.matrix[0].re, g.matrix[0].im));
            c.paired = true;
        } else if (g.kind == QM_BATCH_DIAG) {
            for (u32 i = 0; i < d; ++i) m.push_back(cx(g.matrix[i].re, g.matrix[i].im));
            cv.diagonal(q, m);
        } else {
            for (u32 i = 0; i < d * d; ++i) m.push_back(cx(g.matrix[i].re, g.matrix[i].im));
            if (density && k == 2 && q[1] == q[0] + n / 2) c.paired = true;
            cv.dense(q, std::move(m));
        }
    }
    cv.finish();
    reduce_matrices(c.ops, c.ne);
    return true;
}

}  // namespace
}  // namespace qm
