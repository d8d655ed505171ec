// Tiles of the two-step launches that march along z (k_step2z_fp32,
// k_step2z_fp64): LDS rings and z ranges.
#pragma once

#include "ch4g_planes.h"

namespace ch4g {

// Two steps per launch for 3-D lattices (NZ > 1), marching along z.  A block
// owns a TX x TY column of x-y tiles over a range of zc planes and has one
// thread per node of the tile with its one-node x-y halo.  Iteration j:
//   A  step 1 at plane j for the tile + halo nodes (gather from the global
//      state, collision); the populations with c_z = -1 go to the LDS ring M;
//   B  step 2 at plane j - 1 for the tile nodes, gathering from LDS: c_z = +1
//      from plane j - 2 (ring P), c_z = 0 from plane j - 1 (ring Z), c_z = -1
//      from plane j (ring M); collision into the global output;
//   C  (HOLD) the registers of step A go to ring Z (c_z = 0 and the step-1
//      temperature, the lag of step 2) and ring P (c_z = +1, two slots by
//      plane parity); without HOLD step A writes them at once into the slots
//      step B does not read.
// The tile nodes also keep their populations 16 and 18 (c_z = -1) in ring W,
// which the wall rules of step B read at the node itself one plane later
// (fluid bounce-back at y = 0 takes f_16, f_18 there, the fixed-T rule at
// y = NY - 1 takes g_16, g_18).  Planes just below and above the block's range
// are computed in step A (z halo) but not written.  Per two steps the state is
// read (1 + 2/zc) times over the tile + halo area (M/T of the tile) and
// written once; the temperature lag is read from tl_in and written to tl_out
// (halo nodes of one block are tile nodes of another).
namespace z2 {
// index of population q within its c_z class: c_z = 0: {0,1,2,3,4,7,8,9,10},
// c_z = +1: {5,11,12,15,17}, c_z = -1: {6,13,14,16,18}
__host__ __device__ constexpr int slot(int q)
{
    constexpr int v[Q] = {0, 1, 2, 3, 4, 0, 0, 5, 6, 7, 8, 1, 2, 1, 2, 3, 3, 4, 4};
    return v[q];
}
// ring W index of population 16 / 18
__host__ __device__ constexpr int wslot(int q) { return q == 16 ? 0 : 1; }
}  // namespace z2

// LDS rings of a z-marching tile of TX x TY nodes (one-node x-y halo).
// HOLD: step A keeps its c_z >= 0 results in registers until step C (one
// slot of ring Z, two of ring P, one of ring W); otherwise step A writes
// every result at once into rings with one more slot each (two of Z, three
// of P, two of W).
template <bool FLUID, bool THERMAL, int TX_, int TY_, bool HOLD_>
struct TileZ {
    static constexpr int TX = TX_, TY = TY_, W = TX + 2;
    static constexpr bool HOLD = HOLD_;
    static constexpr int M = W * (TY + 2);            // tile + halo nodes
    static constexpr int T = TX * TY;                 // tile nodes
    static constexpr int THREADS = (M + 63) / 64 * 64;
    static constexpr int F = FLUID ? 1 : 0, H = THERMAL ? 1 : 0;
    static constexpr int KM = 5 * F + 5 * H;          // ring M planes
    static constexpr int KZ = 9 * F + 9 * H + H;      // planes of one ring Z slot (+ lag)
    static constexpr int KP = 5 * F + 5 * H;          // planes of one ring P slot
    static constexpr int KW = 2 * F + 2 * H;          // planes of one ring W slot (tile nodes)
    static constexpr int NZS = HOLD ? 1 : 2, NPS = HOLD ? 2 : 3, NWS = HOLD ? 1 : 2;
    static constexpr int OZ = KM, OP = KM + NZS * KZ, OW = (KM + NZS * KZ + NPS * KP) * M;
    static constexpr int REALS = OW + NWS * KW * T;
    static_assert(THREADS >= T && THREADS <= 1024, "z-marching block");
    // plane of population q (fluid: gq = 0, temperature: gq = 1) in its ring
    static __device__ constexpr int pm(int q, int gq) { return gq * 5 * F + z2::slot(q); }
    static __device__ constexpr int pz(int q, int gq, int s) { return OZ + s * KZ + gq * 9 * F + z2::slot(q); }
    static __device__ constexpr int lag(int s) { return OZ + s * KZ + 9 * F + 9 * H; }
    static __device__ constexpr int pp(int q, int gq, int s) { return OP + s * KP + gq * 5 * F + z2::slot(q); }
    static __device__ constexpr int pw(int q, int gq, int s) { return s * KW + gq * 2 * F + z2::wslot(q); }
};

// Ring slots read by step B at iteration it (plane p = it - 1 of the
// iteration count): ring Z and W of plane p, ring P of plane p and p - 1.
template <class TZ>
struct RingSlots {
    int z, w, p_own, p_below;
    __device__ RingSlots(int it)
    {
        if constexpr (TZ::HOLD) {
            z = 0;
            w = 0;
            p_own = (it - 1) & 1;
            p_below = it & 1;
        } else {
            z = (it - 1) & 1;
            w = (it - 1) & 1;
            p_own = (it - 1) % 3;
            p_below = (it + 1) % 3;  // (it - 2) mod 3
        }
    }
};

// Step-2 gather of population q (gq = 0 fluid, 1 temperature) at tile node
// `at` (tile + halo index) / `tn` (tile index) from the rings.
template <class TZ, int q, int gq, typename T>
__device__ __forceinline__ T ring_src(const T *t, int at, int tn, const RingSlots<TZ> &rs, bool cross)
{
    constexpr int M = TZ::M;
    T v;
    // pull source in the streaming direction
    const int src = at - cxq(q) - cyq(q) * TZ::W;
    if constexpr (czq(q) > 0)
        v = t[TZ::pp(q, gq, rs.p_below) * M + src];
    else if constexpr (czq(q) < 0)
        v = t[TZ::pm(q, gq) * M + src];
    else
        v = t[TZ::pz(q, gq, rs.z) * M + src];
    if constexpr (cyq(q) != 0) {
        // wall rules: fluid bounce-back takes the opposite population at the
        // node itself, the fixed-T rule the same population there
        constexpr int qs = gq == 0 ? invq(q) : q;
        if (cross) {
            if constexpr (czq(qs) > 0)
                v = t[TZ::pp(qs, gq, rs.p_own) * M + at];
            else if constexpr (czq(qs) < 0)
                v = t[TZ::OW + TZ::pw(qs, gq, rs.w) * TZ::T + tn];
            else
                v = t[TZ::pz(qs, gq, rs.z) * M + at];
        }
    }
    return v;
}

// Step A / C: the results of plane j (iteration it) of node m into the
// rings: c_z = -1 into ring M (always), the others when `rest`.
template <class TZ, bool FLUID, bool THERMAL, typename T>
__device__ __forceinline__ void ring_put(T *t, int m, int it, const T rf[Q], const T rg[Q], T rt,
                                         bool tile, int tn, bool minus, bool rest)
{
    constexpr int M = TZ::M;
    const int sz = TZ::HOLD ? 0 : (it & 1), sw = sz;
    const int sp = TZ::HOLD ? (it & 1) : (it % 3);
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (czq(q) < 0) {
            if (minus) {
                if constexpr (FLUID) t[TZ::pm(q, 0) * M + m] = rf[q];
                if constexpr (THERMAL) t[TZ::pm(q, 1) * M + m] = rg[q];
            }
        } else if constexpr (czq(q) == 0) {
            if (rest) {
                if constexpr (FLUID) t[TZ::pz(q, 0, sz) * M + m] = rf[q];
                if constexpr (THERMAL) t[TZ::pz(q, 1, sz) * M + m] = rg[q];
            }
        } else {
            if (rest) {
                if constexpr (FLUID) t[TZ::pp(q, 0, sp) * M + m] = rf[q];
                if constexpr (THERMAL) t[TZ::pp(q, 1, sp) * M + m] = rg[q];
            }
        }
    });
    if (rest) {
        if constexpr (THERMAL) t[TZ::lag(sz) * M + m] = rt;
        if (tile) {
            if constexpr (FLUID) {
                t[TZ::OW + TZ::pw(16, 0, sw) * TZ::T + tn] = rf[16];
                t[TZ::OW + TZ::pw(18, 0, sw) * TZ::T + tn] = rf[18];
            }
            if constexpr (THERMAL) {
                t[TZ::OW + TZ::pw(16, 1, sw) * TZ::T + tn] = rg[16];
                t[TZ::OW + TZ::pw(18, 1, sw) * TZ::T + tn] = rg[18];
            }
        }
    }
}

// z ranges: a CU holds one block (LDS), and a block of zc planes takes zc + 2
// iterations of the same length, so the launch takes ceil(blocks / 256) (zc +
// 2) of them: the most ranges that 1 to 8 full rounds of blocks hold, whichever
// makes this least.  us per step, at least 1024 blocks of at most 128 planes
// (before) -> this: channel 128^3 49.8 -> 47.6 (16 planes), 192^3 188 -> 158
// (28); Rayleigh-Benard 128^3 93.4 -> 89.5, 192^3 351 -> 302, 256^3 703 -> 658
// (128), 320^3 1543 -> 1410, 192x120x280 323 -> 288 (26), 320x100x90 168 ->
// 138 (13), 512^3 5640 -> 5640 (256); double arithmetic 256^3 975 -> 911.
inline int z_range(int64_t columns, int NZ)
{
    constexpr int64_t CUS = 256;
    int64_t best = 0, zbest = NZ;
    for (int64_t round = 1; round <= 8; round++) {
        const int64_t most = (NZ + 3) / 4, fit = round * CUS / columns;
        const int64_t r = fit < 1 ? 1 : (fit > most ? most : fit);
        const int64_t zc = (NZ + r - 1) / r, blocks = columns * ((NZ + zc - 1) / zc);
        const int64_t cost = (blocks + CUS - 1) / CUS * (zc + 2);
        // (more blocks even out the rounds: taken at half a percent more)
        if (round == 1 || cost * 200 <= best * 201) {
            best = cost;
            zbest = zc;
        }
    }
    return (int)zbest;
}

// iterations a launch of that many columns takes with ranges of zc planes
inline int64_t z_iterations(int64_t columns, int NZ, int64_t zc)
{
    return (columns * ((NZ + zc - 1) / zc) + 255) / 256 * (zc + 2);
}

}  // namespace ch4g
