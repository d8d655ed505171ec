// Population planes addressed through buffer resources, and the pull sources
// of a node as byte offsets (device code shared by the step kernels).
#pragma once

#include "ch4g_internal.h"

namespace ch4g {

// The Q planes of a population array as three buffer resources of up to
// seven planes each: a plane is addressed by the resource of its group, a
// scalar offset of its place in the group and the node's 32-bit byte offset
// (planes of less than 4 GiB / 7, planes_ok).  Keeps the scalar registers
// free of 38 64-bit plane addresses and the vector registers of 64-bit lane
// addresses: without them the FP64 step kernel ran 130 64-bit address
// additions and 455 moves of spilled scalars per wave.
template <typename T>
struct Planes {
    __amdgpu_buffer_rsrc_t r[3];
    uint32_t pb;  // plane stride in bytes
};

inline bool planes_ok(const KParams &P, int64_t rsz) { return 7 * P.S * rsz < (int64_t)1 << 32; }

// base: the same in every lane (made so: a batched launch loads it from a table)
template <typename T>
__device__ __forceinline__ Planes<T> make_planes(const T *base, int64_t S)
{
    Planes<T> p;
    const uint64_t b = (uint64_t)base;
    const uint64_t ub = (uint64_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b) & 0xffffffffu,
                   uh = (uint64_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32;
    const uint32_t pb = __builtin_amdgcn_readfirstlane((int)(uint32_t)(S * (int64_t)sizeof(T)));
    p.pb = pb;
    static_for<0, 3>([&](auto gc) {
        constexpr int gi = decltype(gc)::value;
        constexpr int np = gi < 2 ? 7 : Q - 14;
        p.r[gi] = __builtin_amdgcn_make_buffer_rsrc((void *)((uh | ub) + (uint64_t)gi * 7 * pb), (short)0,
                                                    (int)(uint32_t)((uint64_t)np * pb), 0x00020000);
    });
    return p;
}

// cache-policy bits of buffer instructions: non-temporal
constexpr int CPOL_NT = 2;

// voff: per lane; soff: scalar, on top of the place of `plane` in its group
template <int plane, typename T>
__device__ __forceinline__ T plane_load(const Planes<T> &p, uint32_t voff, uint32_t soff)
{
    const int s = (int)((uint32_t)(plane % 7) * p.pb + soff);
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(p.r[plane / 7], (int)voff, s, 0));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(p.r[plane / 7], (int)voff, s, 0));
}

template <int plane, bool NT, typename T>
__device__ __forceinline__ void plane_store(const Planes<T> &p, uint32_t voff, uint32_t soff, T v)
{
    const int s = (int)((uint32_t)(plane % 7) * p.pb + soff);
    if constexpr (sizeof(T) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), p.r[plane / 7], (int)voff, s,
                                              NT ? CPOL_NT : 0);
    } else {
        typedef uint32_t u2 __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), p.r[plane / 7], (int)voff, s,
                                              NT ? CPOL_NT : 0);
    }
}

// Byte offsets within a plane of the coordinates a node pulls from: x[1 + c]
// that of x - c, likewise y and z.  UNI: what the wave shares goes into the
// scalar offset of the loads (PULL_ROW: y and z, PULL_LINEAR: nothing).
enum { PULL_LINEAR = 0, PULL_ROW = 1 };
template <typename T, int UNI>
struct Pull {
    uint32_t x[3], y[3], z[3];
    __device__ Pull(const Nbr &b, int NX, int NY)
    {
        constexpr uint32_t B = sizeof(T);
        const uint32_t row = B * (uint32_t)NX, plane = row * (uint32_t)NY;
        x[0] = B * (uint32_t)b.xp;
        x[1] = B * (uint32_t)b.x;
        x[2] = B * (uint32_t)b.xm;
        y[0] = row * (uint32_t)b.yp;
        y[1] = row * (uint32_t)b.y;
        y[2] = row * (uint32_t)b.ym;
        z[0] = plane * (uint32_t)b.zp;
        z[1] = plane * (uint32_t)b.z;
        z[2] = plane * (uint32_t)b.zm;
    }
    // parts of the source of population q (q = 0: the node itself)
    template <int q>
    __device__ uint32_t voff() const
    {
        return UNI == PULL_ROW ? x[1 + cxq(q)] : x[1 + cxq(q)] + y[1 + cyq(q)] + z[1 + czq(q)];
    }
    template <int q>
    __device__ uint32_t soff() const
    {
        return UNI == PULL_ROW ? y[1 + cyq(q)] + z[1 + czq(q)] : 0u;
    }
    // plane `base` + d at the source of q, or + dc at the node itself where
    // the lane's (PULL_ROW: the wave's) source lies behind a wall
    template <int q, int base>
    __device__ T load(const Planes<T> &p, bool cross, uint32_t d, uint32_t dc) const
    {
        if constexpr (UNI == PULL_ROW)
            return plane_load<base>(p, cross ? voff<0>() : voff<q>(), cross ? soff<0>() + dc : soff<q>() + d);
        else
            return plane_load<base>(p, cross ? voff<0>() + dc : voff<q>() + d, 0u);
    }
};

// fluid source of population q: x - c_q, or behind a wall the opposite
// population of the node itself (halfway bounce-back)
template <int q, typename T, int UNI>
__device__ __forceinline__ T pull_fluid(const Planes<T> &p, const Pull<T, UNI> &o, bool cross)
{
    if constexpr (cyq(q) == 0) {
        return plane_load<q>(p, o.template voff<q>(), o.template soff<q>());
    } else {
        constexpr int iq = q % 7, ii = invq(q) % 7, mn = iq < ii ? iq : ii;
        static_assert(q / 7 == invq(q) / 7, "opposite planes share a resource");
        return o.template load<q, q / 7 * 7 + mn>(p, cross, (uint32_t)(iq - mn) * p.pb, (uint32_t)(ii - mn) * p.pb);
    }
}

// temperature source of population q: x - c_q, or behind a wall the same
// population of the node itself (fixed-temperature rule)
template <int q, typename T, int UNI>
__device__ __forceinline__ T pull_thermal(const Planes<T> &p, const Pull<T, UNI> &o, bool cross)
{
    if constexpr (cyq(q) == 0)
        return plane_load<q>(p, o.template voff<q>(), o.template soff<q>());
    else
        return o.template load<q, q>(p, cross, 0u, 0u);
}

// f(std::true_type) or f(std::false_type)
template <typename F>
inline void with_bool(bool v, F &&f)
{
    if (v)
        f(std::true_type{});
    else
        f(std::false_type{});
}

}  // namespace ch4g
