// FP64 fused stream+collide kernel and gather (hydro_fields) kernel.
//
// Arithmetic is written in the reference's evaluation order and this file is
// compiled with -ffp-contract=off (the reference builds with -std=c11, which
// disables contraction), so every field is bit-identical to the reference's
// FP64 step on the same inputs.
//
// State between steps (pull scheme): the post-collision populations of the
// last step (the reference's rhs_p/rhs_g after add_forcing), plus one lag
// scalar per node, tlag = the temperature of the previous step.  The kernel
// for step s first performs the streaming of step s-1 (lb.c:544-583) with the
// wall rules of boundary_conditions.c applied as a gather, reconstructs
// rho, u, T of step s-1 (lb.c:420-540; the u shift uses the force built from
// the lagged temperature, as main.c's ordering implies), then collides
// (fluid.c:1033-1225) and adds the Guo term (forcing.c:1424-1435) of step s.
#include "ch4g_planes.h"
#include "ch4g_ztile.h"

namespace ch4g {

// typedef.h:286-291, strict left-to-right sums
__device__ __forceinline__ double m_sum(const double *p)
{
    return p[0] + p[1] + p[2] + p[3] + p[4] + p[5] + p[6] + p[7] + p[8] + p[9] + p[10] + p[11] + p[12] + p[13] +
           p[14] + p[15] + p[16] + p[17] + p[18];
}
__device__ __forceinline__ double m_x(const double *p)
{
    return p[1] - p[2] + p[7] + p[8] - p[9] - p[10] + p[11] - p[12] + p[13] - p[14];
}
__device__ __forceinline__ double m_y(const double *p)
{
    return p[3] - p[4] + p[7] - p[8] + p[9] - p[10] + p[15] + p[16] - p[17] - p[18];
}
__device__ __forceinline__ double m_z(const double *p)
{
    return p[5] - p[6] + p[11] + p[12] - p[13] - p[14] + p[15] - p[16] + p[17] - p[18];
}

// build_forcing for one node (forcing.c:361-667), terms added in source order;
// with NOZEROMODE the mean of those terms is removed (forcing.c:1123-1152)
// before the particle feedback is added (main.c:118-131).  GEN: the HIT,
// NOZEROMODE and two-way terms are compiled in (with the LES closures of the
// step); lattices without them run an instance without their registers.
template <bool GEN = true>
__device__ __forceinline__ void force_at(const KParams &P, const HitTable &tab, const double *fb, const double *f0,
                                         uint32_t n, int x, int y, int z, double T, double F[3])
{
    F[0] = P.Fc[0];
    F[1] = P.Fc[1];
    F[2] = P.Fc[2];
    if (GEN && P.hit) {
#pragma unroll
        for (int ii = 0; ii < CH4G_HIT_NK; ii++) {
            double ax = tab.sx[ii * P.NX + x];
            double ay = tab.sy[ii * P.NY + y];
            double az = tab.sz[ii * P.NZ + z];
            F[0] += P.hit_fa[0][ii] * (ay + az);
            F[1] += P.hit_fa[1][ii] * (ax + az);
            F[2] += P.hit_fa[2][ii] * (ay + ax);
        }
    }
    if (P.buoy) {
        double temp = T - P.T0b;
        double fac = P.beta_t * temp;
        if (P.beta2_t != 0.0) fac += P.beta2_t * temp * temp;
        F[0] += fac * P.grav[0];
        F[1] += fac * P.grav[1];
        F[2] += fac * P.grav[2];
    }
    if (GEN && f0) {
        F[0] -= f0[0];
        F[1] -= f0[1];
        F[2] -= f0[2];
    }
    if (GEN && P.twoway) {
        const size_t N = (size_t)P.N;
        F[0] += fb[n];
        F[1] += fb[N + n];
        F[2] += fb[2 * N + n];
    }
}

// Streaming of the previous step as a pull, with halfway bounce-back at y
// walls (boundary_conditions.c:714-873: the ghost receives the node's own
// post-collision population of the opposite direction).  Branch-free so all
// loads are in flight together.
template <bool FIRST>
__device__ __forceinline__ void gather_fluid(const KParams &P, const Nbr &b, const double *__restrict__ in,
                                             uint32_t n, double f[Q])
{
    const size_t N = (size_t)P.S;  // plane stride
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (FIRST) {
            f[q] = in[(size_t)q * N + n];
        } else {
            const bool cross = P.wall_f && crosses_wall<q>(b);
            const double *base = in + (size_t)(cross ? invq(q) : q) * N;
            const uint32_t off = cross ? n : src_index<q>(b, P.NX, P.NY);
            f[q] = base[off];
        }
    });
}

// Fixed-temperature y walls (boundary_conditions.c:966-1078): the ghost
// receives the node's own post-collision population of the SAME direction
// plus w_q * 2((T_wall - T_ref) - t), t being the node temperature of the
// previous hydro_fields call (the lag scalar).
template <bool FIRST>
__device__ __forceinline__ void gather_thermal(const KParams &P, const Nbr &b, const double *__restrict__ in,
                                               uint32_t n, double Tlag, double g[Q])
{
    const size_t N = (size_t)P.S;  // plane stride
    const double fac_top = 2.0 * (P.Tw_top - Tlag);
    const double fac_bot = 2.0 * (P.Tw_bot - Tlag);
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (FIRST) {
            g[q] = in[(size_t)q * N + n];
        } else {
            const bool cross = P.wall_t && crosses_wall<q>(b);
            const uint32_t off = cross ? n : src_index<q>(b, P.NX, P.NY);
            const double v = in[(size_t)q * N + off];
            if constexpr (cyq(q) > 0)
                g[q] = cross ? v + wq(q) * fac_bot : v;
            else if constexpr (cyq(q) < 0)
                g[q] = cross ? v + wq(q) * fac_top : v;
            else
                g[q] = v;
        }
    });
}

// the same gathers through buffer resources
template <int UNI>
__device__ __forceinline__ void pull_fluid64(const KParams &P, const Nbr &b, const Planes<double> &in,
                                             const Pull<double, UNI> &o, double f[Q])
{
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = pull_fluid<q>(in, o, P.wall_f && crosses_wall<q>(b));
    });
}

template <int UNI>
__device__ __forceinline__ void pull_thermal64(const KParams &P, const Nbr &b, const Planes<double> &in,
                                               const Pull<double, UNI> &o, double Tlag, double g[Q])
{
    const double fac_top = 2.0 * (P.Tw_top - Tlag);
    const double fac_bot = 2.0 * (P.Tw_bot - Tlag);
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const bool cross = P.wall_t && crosses_wall<q>(b);
        const double v = pull_thermal<q>(in, o, cross);
        if constexpr (cyq(q) > 0)
            g[q] = cross ? v + wq(q) * fac_bot : v;
        else if constexpr (cyq(q) < 0)
            g[q] = cross ? v + wq(q) * fac_top : v;
        else
            g[q] = v;
    });
}

// Where a node's populations go, through buffer resources or (flat) plane
// pointers; non-temporal (NT) where step_order says so.
template <bool NT, int UNI>
struct PlaneOut {
    Planes<double> p;
    Pull<double, UNI> o;
    template <int q>
    __device__ void put(double v) const
    {
        plane_store<q, NT>(p, o.template voff<0>(), o.template soff<0>(), v);
    }
};
template <bool NT>
struct FlatOut {
    double *__restrict__ p;
    size_t S;
    uint32_t n;
    template <int q>
    __device__ void put(double v) const
    {
        double *a = p + (size_t)q * S + n;
        if constexpr (NT)
            __builtin_nontemporal_store(v, a);
        else
            *a = v;
    }
};

// equilibrium (lb.c:382-415) of the opposite pair (q, inv q), and c.u of q:
//   rho w (1 + c.u / cs^2 + (c.u)^2 / (2 cs^4) - u^2 / (2 cs^2)),
// in the reference's order.  Products by a velocity component 0 or +-1 are
// left out: c.u is one or two signed terms, and c.u of the opposite direction
// its negative, both exact (an IEEE sum with a zero term, and of negated
// terms, is the same number; the sign of a zero c.u cannot reach the result).
// The zero products do one thing: a velocity that is not finite makes every
// population NaN.  u2z carries that (u2 + 0 ux + 0 uy + 0 uz).
// With the products, the general force paths and 64-bit lane addresses in one
// kernel a wave ran 2068 vector instructions (1473 FP64) per node; this
// instance 751 (680).  us per step: Rayleigh-Benard 256x128 9.8 -> 6.1,
// 512x256 14.8 -> 12.7, 64^3 25.6 -> 24.1; channel 4x64x4 4.56 -> 3.83, 64^3
// 14.5 -> 12.8; larger lattices are bound by memory and stay (256^3 1.0 x).
template <int q>
__device__ __forceinline__ double cdot64(double x, double y, double z)
{
    constexpr int a = cxq(q), b = cyq(q), c = czq(q);
    const double tx = a > 0 ? x : -x, ty = b > 0 ? y : -y, tz = c > 0 ? z : -z;
    if constexpr (a != 0 && b != 0)
        return tx + ty;
    else if constexpr (a != 0 && c != 0)
        return tx + tz;
    else if constexpr (b != 0 && c != 0)
        return ty + tz;
    else
        return a != 0 ? tx : (b != 0 ? ty : tz);
}

__device__ __forceinline__ double u2_of(double ux, double uy, double uz)
{
    const double u2 = (ux * ux + uy * uy + uz * uz);
    return u2 + (0.0 * ux + 0.0 * uy + 0.0 * uz);
}

// representative q of the k-th opposite pair
__host__ __device__ constexpr int pair64(int k)
{
    constexpr int v[9] = {1, 3, 5, 7, 8, 11, 12, 15, 16};
    return v[k];
}

struct EqPair {
    double cu, eq, eqb;  // c_q.u, equilibrium of q and of inv q
};
template <int q>
__device__ __forceinline__ EqPair feq_pair(const KParams &P, double rho, double ux, double uy, double uz, double u2z)
{
    EqPair e;
    e.cu = cdot64<q>(ux, uy, uz);
    const double a = P.invcs2 * e.cu, b = P.invtwocs4 * e.cu * e.cu, c = P.invtwocs2 * u2z, rw = rho * wq(q);
    e.eq = rw * (1.0 + a + b - c);
    e.eqb = rw * (1.0 - a + b - c);
    return e;
}
__device__ __forceinline__ double feq_rest(const KParams &P, double rho, double u2z)
{
    return rho * wq(0) * (1.0 - P.invtwocs2 * u2z);
}

// tau_u_les, local-strain branch (les.c:20-30,:144-180,:253) with the
// stress_tensor assignments of gradients.c:42-69.
__device__ __forceinline__ double les_tau(const KParams &P, const double f[Q], double rho, double ux, double uy,
                                          double uz, double u2z, double tau_prev)
{
    double d[Q];
    static_for<0, 9>([&](auto kk) {
        constexpr int q = pair64(decltype(kk)::value), qb = invq(q);
        const EqPair e = feq_pair<q>(P, rho, ux, uy, uz, u2z);
        d[q] = f[q] - e.eq;
        d[qb] = f[qb] - e.eqb;
    });
    // sums over q in order; terms with a zero factor left out as above
    double xx = 0.0, yy = 0.0, xy = 0.0, xz = 0.0, yz = 0.0;
    static_for<1, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value, cx = cxq(q), cy = cyq(q), cz = czq(q);
        if constexpr (cx != 0) xx += d[q];
        if constexpr (cy != 0) yy += d[q];
        if constexpr (cx * cy != 0) xy += cx * cy > 0 ? d[q] : -d[q];
        if constexpr (cx * cz != 0) xz += cx * cz > 0 ? d[q] : -d[q];
        if constexpr (cy * cz != 0) yz += cy * cz > 0 ? d[q] : -d[q];
    });
    const double yx = xy, zx = 0.0, zy = yz;
    const double zz = xz;
    double fac = -1.0 / (2 * P.cs2 * rho * tau_prev * 1.0);
    double s_norm = fabs(fac) * sqrt(2.0 * (xx * xx + xy * xy + xz * xz + yx * yx + yy * yy + yz * yz + zx * zx +
                                            zy * zy + zz * zz));
    double nu_les = s_norm * P.Cs2;
    return 3.0 * (nu_les + P.nu) + 0.5;
}

// tau_u_les, default finite-difference branch (les.c:31-43, :160-180, :253):
// gradient_vector of the stored velocity (gradients.c:78-499: centred
// differences with periodic images, one-sided second order at y walls,
// components along a size-one axis zeroed), |S| = sqrt(2 S_ij S_ij) summed
// in the reference's term order.  tens.ab = d u_a / d x_b.
__device__ __forceinline__ double les_tau_fd(const KParams &P, const double *__restrict__ vel, const Nbr &b,
                                             uint32_t n)
{
    const size_t N = (size_t)P.N;
    const int NX = P.NX, NY = P.NY;
    auto id = [&](int i, int j, int k) -> size_t { return ((size_t)k * NY + j) * NX + i; };
    double G[3][3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const double *u = vel + c * N;
        G[c][0] = (u[id(b.xp, b.y, b.z)] - u[id(b.xm, b.y, b.z)]) / 2.0;
        G[c][1] = (u[id(b.x, b.yp, b.z)] - u[id(b.x, b.ym, b.z)]) / 2.0;
        G[c][2] = (u[id(b.x, b.y, b.zp)] - u[id(b.x, b.y, b.zm)]) / 2.0;
        if (P.wall_f) {
            if (b.bot) G[c][1] = -1.5 * u[n] + 2.0 * u[id(b.x, 1, b.z)] + -0.5 * u[id(b.x, 2, b.z)];
            if (b.top) G[c][1] = 1.5 * u[n] + -2.0 * u[id(b.x, NY - 2, b.z)] + 0.5 * u[id(b.x, NY - 3, b.z)];
        }
        if (P.NX == 1) G[c][0] = 0.0;
        if (NY == 1) G[c][1] = 0.0;
        if (P.NZ == 1) G[c][2] = 0.0;
    }
    const double xx = G[0][0], xy = G[0][1], xz = G[0][2];
    const double yx = G[1][0], yy = G[1][1], yz = G[1][2];
    const double zx = G[2][0], zy = G[2][1], zz = G[2][2];
    double s_norm = sqrt(0.5 * ((xx + xx) * (xx + xx) + (xy + yx) * (xy + yx) + (xz + zx) * (xz + zx) +
                                (yx + xy) * (yx + xy) + (yy + yy) * (yy + yy) + (yz + zy) * (yz + zy) +
                                (zx + xz) * (zx + xz) + (zy + yz) * (zy + yz) + (zz + zz) * (zz + zz)));
    double nu_les = s_norm * P.Cs2;
    return 3.0 * (nu_les + P.nu) + 0.5;
}

// tau_t_les (les.c:273-297, METHOD_STREAMING, prandtl = 1.0)
__device__ __forceinline__ double les_tau_t(const KParams &P, double tau_les)
{
    const double prandtl = 1.0;
    return 3.0 * (P.kappa + (tau_les - 0.5 - 3 * P.nu) / (3 * prandtl)) + 0.5;
}

// hydro_fields of the previous step for one node (lb.c:420-540): density and
// velocity with the half force built from the lagged temperature.
template <bool GEN = true>
__device__ __forceinline__ void fluid_velocity64(const KParams &P, const double f[Q], uint32_t n, int x, int y, int z,
                                                 double Tlag, double &rho, double &ux, double &uy, double &uz)
{
    rho = m_sum(f);
    if (P.forced) {
        double Fp[3];
        force_at<GEN>(P, P.hit_prev, P.fb_prev, P.f0p, n, x, y, z, Tlag, Fp);
        ux = m_x(f) / rho + 0.5 * 1.0 * Fp[0];
        uy = m_y(f) / rho + 0.5 * 1.0 * Fp[1];
        uz = m_z(f) / rho + 0.5 * 1.0 * Fp[2];
    } else {
        ux = m_x(f) / rho;
        uy = m_y(f) / rho;
        uz = m_z(f) / rho;
    }
}

// What the fluid's collision leaves for the temperature's.
struct Moved64 {
    double ux = 0.0, uy = 0.0, uz = 0.0, tau_les = 0.0;
};

// Collision and force of one node's gathered populations, shared by every
// step kernel, so a lattice advances bit-identically in all: the fluid's f...
template <bool GEN, class OutF>
__device__ __forceinline__ void collide_fluid64(const KParams &P, const Nbr &b, const double f[Q], double Tlag, double T,
                                                double *__restrict__ taules, uint32_t n, const OutF &outf, Moved64 &mv)
{
    const int x = b.x, y = b.y, z = b.z;
    double &ux = mv.ux, &uy = mv.uy, &uz = mv.uz, &tau_les = mv.tau_les;
    double rho;
    fluid_velocity64<GEN>(P, f, n, x, y, z, Tlag, rho, ux, uy, uz);
    const double u2z = u2_of(ux, uy, uz);
    double invtau = P.invtau_u;
    if (GEN && P.les) {
        if (P.les_fd) {
            tau_les = les_tau_fd(P, (const double *)P.vel, b, n);
        } else {
            double tau_prev = (P.itime == 1) ? P.tau_u : taules[n];
            tau_les = les_tau(P, f, rho, ux, uy, uz, u2z, tau_prev);
        }
        taules[n] = tau_les;
        invtau = 1.0 / tau_les;
    }
    double Fn[3] = {0.0, 0.0, 0.0};
    if (P.forced) force_at<GEN>(P, P.hit_now, P.fb_now, P.f0n, n, x, y, z, T, Fn);
    // r += guo w rho F . ((c - u) / cs^2 + c (c.u) / cs^4), components in
    // order; s = +1 for q, -1 for its opposite (c (c.u) is the same for both)
    const double gf[3] = {P.guo_fac * wq(0) * rho, P.guo_fac * wq(1) * rho, P.guo_fac * wq(7) * rho};
    auto guo = [&](auto qc, double s, double cc, double &r) {
        constexpr int q = decltype(qc)::value, wc = q == 0 ? 0 : (q <= 6 ? 1 : 2);
        constexpr int c[3] = {cxq(q), cyq(q), czq(q)};
        const double u[3] = {ux, uy, uz};
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const double ca = c[a] * s;  // 0 or +-1, known at compile time
            double d = (ca - u[a]) * P.invcs2;
            if (c[a] != 0) d += c[a] > 0 ? cc : -cc;
            r += gf[wc] * Fn[a] * d;
        }
    };
    {
        double r = f[0];
        r += -invtau * (f[0] - feq_rest(P, rho, u2z));
        if (P.forced) guo(std::integral_constant<int, 0>{}, 1.0, 0.0, r);
        outf.template put<0>(r);
    }
    static_for<0, 9>([&](auto kk) {
        constexpr int q = pair64(decltype(kk)::value), qb = invq(q);
        const EqPair e = feq_pair<q>(P, rho, ux, uy, uz, u2z);
        double r = f[q], rb = f[qb];
        r += -invtau * (f[q] - e.eq);
        rb += -invtau * (f[qb] - e.eqb);
        if (P.forced) {
            const double cc = e.cu * P.invcs4;
            guo(std::integral_constant<int, q>{}, 1.0, cc, r);
            guo(std::integral_constant<int, q>{}, -1.0, cc, rb);
        }
        outf.template put<q>(r);
        outf.template put<qb>(rb);
    });
}

// ... and the temperature's g, of sum T.
template <bool FLUID, bool GEN, class OutG>
__device__ __forceinline__ void collide_thermal64(const KParams &P, const double g[Q], double T, const Moved64 &mv,
                                                  const OutG &outg)
{
    const double ux = mv.ux, uy = mv.uy, uz = mv.uz, tau_les = mv.tau_les;
    const double u2z = u2_of(ux, uy, uz);
    double invtau_t = P.invtau_t;
    if constexpr (FLUID)
        if (GEN && P.les_t) invtau_t = 1.0 / les_tau_t(P, tau_les);
    {
        double r = g[0];
        r += -invtau_t * (g[0] - feq_rest(P, T, u2z));
        outg.template put<0>(r);
    }
    static_for<0, 9>([&](auto kk) {
        constexpr int q = pair64(decltype(kk)::value), qb = invq(q);
        const EqPair e = feq_pair<q>(P, T, ux, uy, uz, u2z);
        double r = g[q], rb = g[qb];
        r += -invtau_t * (g[q] - e.eq);
        rb += -invtau_t * (g[qb] - e.eqb);
        outg.template put<q>(r);
        outg.template put<qb>(rb);
    });
}

template <bool FLUID, bool THERMAL, bool GEN, class OutF, class OutG>
__device__ __forceinline__ void collide64(const KParams &P, const Nbr &b, const double f[Q], const double g[Q],
                                          double Tlag, double T, double *__restrict__ taules, uint32_t n,
                                          const OutF &outf, const OutG &outg)
{
    Moved64 mv;
    if constexpr (FLUID) collide_fluid64<GEN>(P, b, f, Tlag, T, taules, n, outf, mv);
    if constexpr (THERMAL) collide_thermal64<FLUID, GEN>(P, g, T, mv, outg);
}

// One node of the fused step.  UNI: what the wave shares (Pull).  BUF: planes
// through buffer resources (planes_ok), else through pointers.
template <bool FIRST, bool FLUID, bool THERMAL, bool NT, bool GEN, bool BUF, int UNI>
__device__ __forceinline__ void step_node64(const KParams &P, const double *__restrict__ fin,
                                            const double *__restrict__ gin, double *__restrict__ fout,
                                            double *__restrict__ gout, double *__restrict__ tlag,
                                            double *__restrict__ taules, int x, int y, int z, uint32_t n)
{
    const Nbr b = make_nbr(x, y, z, P.NX, P.NY, P.NZ);
    double Tlag = 0.0, T = 0.0;
    double g[Q], f[Q];
    if constexpr (THERMAL) Tlag = tlag[n];
    if constexpr (BUF) {
        static_assert(!FIRST, "the first step reads pre-collision populations");
        const Pull<double, UNI> o(b, P.NX, P.NY);
        if constexpr (THERMAL) pull_thermal64(P, b, make_planes(gin, P.S), o, Tlag, g);
        if constexpr (FLUID) pull_fluid64(P, b, make_planes(fin, P.S), o, f);
        if constexpr (THERMAL) T = m_sum(g);
        const PlaneOut<NT, UNI> outf{make_planes(FLUID ? fout : gout, P.S), o};
        const PlaneOut<NT, UNI> outg{make_planes(THERMAL ? gout : fout, P.S), o};
        collide64<FLUID, THERMAL, GEN>(P, b, f, g, Tlag, T, taules, n, outf, outg);
    } else {
        if constexpr (THERMAL) gather_thermal<FIRST>(P, b, gin, n, Tlag, g);
        if constexpr (FLUID) gather_fluid<FIRST>(P, b, fin, n, f);
        if constexpr (THERMAL) T = m_sum(g);
        collide64<FLUID, THERMAL, GEN>(P, b, f, g, Tlag, T, taules, n, FlatOut<NT>{fout, (size_t)P.S, n},
                                       FlatOut<NT>{gout, (size_t)P.S, n});
    }
    if constexpr (THERMAL) tlag[n] = T;
}

// Row grid or, DENSE, a linear grid with one node per lane (see dense_rows),
// in the block order of step_order.
template <bool FIRST, bool FLUID, bool THERMAL, bool DENSE, bool NT, bool GEN, bool BUF>
__global__ void __launch_bounds__(256) k_step_fp64(KParams P, const double *__restrict__ fin,
                                                   const double *__restrict__ gin, double *__restrict__ fout,
                                                   double *__restrict__ gout, double *__restrict__ tlag,
                                                   double *__restrict__ taules, int run)
{
    int x, y, z;
    uint32_t n;
    const uint32_t lb = xcd_run(run, block_linear(), gridDim.x * gridDim.y * gridDim.z);
    if constexpr (DENSE) {
        n = lb * blockDim.x + threadIdx.x;
        if (n >= (uint32_t)P.N) return;
        const uint32_t row = n / (uint32_t)P.NX;
        x = (int)(n - row * (uint32_t)P.NX);
        y = (int)(row % (uint32_t)P.NY);
        z = (int)(row / (uint32_t)P.NY);
    } else {
        const uint32_t row = lb / gridDim.x;
        x = (lb - row * gridDim.x) * blockDim.x + threadIdx.x;
        if (x >= P.NX) return;
        y = (int)(row % (uint32_t)P.NY);
        z = (int)(row / (uint32_t)P.NY);
        n = row * (uint32_t)P.NX + x;
    }
    step_node64<FIRST, FLUID, THERMAL, NT, GEN, BUF, DENSE ? PULL_LINEAR : PULL_ROW>(P, fin, gin, fout, gout, tlag, taules, x, y, z, n);
}

// Results of a node kept in registers (step A of k_step2z_fp64)
struct RegOut64 {
    double *__restrict__ r;
    template <int q>
    __device__ void put(double v) const
    {
        r[q] = v;
    }
};

// Two steps per launch for 3-D lattices: k_step2z_fp32's march along z
// (ch4g_ztile.h) with this file's arithmetic, so the same bits as two single
// steps.
//
// A single step moves the state at 5 TB/s and is bound by that; here it is
// read (with the tile's halo 1.33 times, 1.07 from memory as the L2s share halo
// lines) and written once per two steps.  us
// per step, single -> this: Rayleigh-Benard 96^3 112 -> 81, 128^3 249 -> 186,
// 185^3 752 -> 589, 256^3 1996 -> 1492, 96x80x112 111 -> 83; channel 113^3
// 91 -> 72, 128^3 120 -> 86, 192^3 413 -> 280.  An iteration (11.6 us at 256^3)
// is now loads, collision, barrier, collision and stores in turn, one block
// per CU: bound by their latencies.  us per step at 256^3 of what did not
// help: the temperature's populations gathered once in step B (9 registers
// spilled) 1564; 64 x 4 tiles 1498 (96^3 98), 32 x 9 1543, 16 x 16 1711, two
// blocks of 16 x 8 per CU 1826; the next plane's loads in flight during B
// (53 registers spilled) 2663, its lines touched ahead 1542.
template <bool FLUID, bool THERMAL, bool NT, class TZ>
__global__ void __launch_bounds__(TZ::THREADS) k_step2z_fp64(KParams P, const double *__restrict__ fin,
                                                             const double *__restrict__ gin, double *__restrict__ fout,
                                                             double *__restrict__ gout,
                                                             const double *__restrict__ tl_in,
                                                             double *__restrict__ tl_out, int zc)
{
    constexpr int M = TZ::M, W = TZ::W, TX = TZ::TX, TY = TZ::TY;
    static_assert(TZ::HOLD, "one slot of ring Z");
    __shared__ double t[TZ::REALS];
    const int NX = P.NX, NY = P.NY, NZ = P.NZ;
    const uint32_t nbx = gridDim.x, nby = gridDim.y;
    const uint32_t bid = xcd_block(block_linear(), nbx * nby * gridDim.z);
    const int x0 = (int)(bid % nbx) * TX, y0 = (int)((bid / nbx) % nby) * TY;
    const int zb = (int)(bid / (nbx * nby)) * zc, ze = min(zb + zc, NZ);
    const int w = NX - x0 < TX ? NX - x0 : TX;
    // step A node of this thread (tile + halo)
    const int m = threadIdx.x, lx = m % W, ly = m / W;
    const bool act_a = m < M && lx <= w + 1;
    int xa = x0 - 1 + lx;
    xa = xa < 0 ? xa + NX : (xa >= NX ? xa - NX : xa);
    int ya = (y0 - 1 + ly) % NY;
    ya = ya < 0 ? ya + NY : ya;
    const bool tile_a = act_a && lx >= 1 && lx <= w && ly >= 1 && ly <= TY;
    const int tn_a = (ly - 1) * TX + (lx - 1);
    // step B node of this thread (tile)
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int xb = x0 + tx, yb = y0 + ty;
    const bool act_b = ty < TY && tx < w && yb < NY;
    const int at = (ty + 1) * W + tx + 1, tn = ty * TX + tx;

    const Planes<double> pin_f = make_planes(FLUID ? fin : gin, P.S), pin_g = make_planes(THERMAL ? gin : fin, P.S);
    const Planes<double> pout_f = make_planes(FLUID ? fout : gout, P.S),
                         pout_g = make_planes(THERMAL ? gout : fout, P.S);
    // step A's node at iteration it (plane zb - 1 + it, periodic in z)
    auto node_a = [&](int it) {
        const int j = zb - 1 + it;
        return make_nbr(xa, ya, j < 0 ? j + NZ : (j >= NZ ? j - NZ : j), NX, NY, NZ);
    };
    auto index = [&](const Nbr &b) { return ((uint32_t)b.z * NY + b.y) * NX + b.x; };
    // the fixed-temperature rule of pull_thermal64
    auto walls = [&](const Nbr &b, double Tlag, double (&g)[Q]) {
        const double fac_top = 2.0 * (P.Tw_top - Tlag);
        const double fac_bot = 2.0 * (P.Tw_bot - Tlag);
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const bool cross = P.wall_t && crosses_wall<q>(b);
            if constexpr (cyq(q) > 0) g[q] = cross ? g[q] + wq(q) * fac_bot : g[q];
            if constexpr (cyq(q) < 0) g[q] = cross ? g[q] + wq(q) * fac_top : g[q];
        });
    };
    const int nit = ze - zb + 2;
    for (int it = 0; it < nit; it++) {
        double rf[Q], rg[Q], rt = 0.0;
        // ---- A: step 1 at plane zb - 1 + it
        if (act_a) {
            const Nbr b = node_a(it);
            const uint32_t n = index(b);
            const Pull<double, PULL_LINEAR> o(b, NX, NY);
            double f[Q], g[Q], Tlag = 0.0;
            if constexpr (THERMAL) {
                Tlag = tl_in[n];
                pull_thermal64(P, b, pin_g, o, Tlag, g);
            }
            if constexpr (FLUID) pull_fluid64(P, b, pin_f, o, f);
            if constexpr (THERMAL) rt = m_sum(g);
            collide64<FLUID, THERMAL, false>(P, b, f, g, Tlag, rt, nullptr, n, RegOut64{rf}, RegOut64{rg});
            ring_put<TZ, FLUID, THERMAL>(t, m, it, rf, rg, rt, tile_a, tn_a, true, false);
        }
        __syncthreads();
        // ---- B: step 2 one plane below (planes of the block's range only)
        const int p = zb - 2 + it;
        if (act_b && p >= zb) {
            const Nbr b = make_nbr(xb, yb, p, NX, NY, NZ);
            const RingSlots<TZ> rs(it);
            const Pull<double, PULL_LINEAR> o(b, NX, NY);
            double Tlag = 0.0, T = 0.0;
            Moved64 mv;
            // read twice, for T and for the collision, so that they hold no
            // registers during the fluid's
            auto g_of = [&](double (&g)[Q]) {
                static_for<0, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    g[q] = ring_src<TZ, q, 1>(t, at, tn, rs, P.wall_t && crosses_wall<q>(b));
                });
                walls(b, Tlag, g);
            };
            if constexpr (THERMAL) {
                double g[Q];
                Tlag = t[TZ::lag(rs.z) * M + at];
                g_of(g);
                T = m_sum(g);
                tl_out[index(b)] = T;
            }
            if constexpr (FLUID) {
                double f[Q];
                static_for<0, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    f[q] = ring_src<TZ, q, 0>(t, at, tn, rs, P.wall_f && crosses_wall<q>(b));
                });
                collide_fluid64<false>(P, b, f, Tlag, T, nullptr, 0u, PlaneOut<NT, PULL_LINEAR>{pout_f, o}, mv);
            }
            if constexpr (THERMAL) {
                asm volatile("" ::: "memory");
                double g[Q];
                g_of(g);
                collide_thermal64<FLUID, false>(P, g, T, mv, PlaneOut<NT, PULL_LINEAR>{pout_g, o});
            }
        }
        __syncthreads();
        // ---- C: the c_z >= 0 results of A into rings Z, P, W
        if (act_a) ring_put<TZ, FLUID, THERMAL>(t, m, it, rf, rg, rt, tile_a, tn_a, false, true);
    }
}

// Two steps per launch for 2-D lattices (k_step2_fp32 with this file's
// arithmetic): the first step of a TX x TY tile and its one-node halo goes
// into LDS, one node per thread, the second from there into the global state.
//
// Small lattices pay one launch's ramp and drain, large ones one read (1.6
// times, with the halo; 1.1 from memory) and write of the state, for two steps.  32 x 4 tiles:
// two blocks of 64 KB of LDS on a CU, so one's loads overlap the other's
// collisions.  us per step, single -> this: Rayleigh-Benard 64x32 3.92 -> 3.56,
// 256x128 6.1 -> 4.2, 512x256 12.5 -> 10.6, 969x487 58.7 -> 39.2, 1024x512 67
// -> 45, 2048x1024 248 -> 152; channel 512x256 7.7 -> 6.4, 1024x512 24.5 ->
// 17.2.  Other tiles at 512x256 and 2048x1024: 16 x 8 10.6 and 161, 32 x 5
// 10.9 and 151, 32 x 8 (one block a CU) 11.7 and 185, 64 x 4 11.7 and 184.
constexpr int T2D_TX = 32, T2D_TY = 4;
template <bool FLUID, bool THERMAL, int TX_, int TY_>
struct Tile2D {
    static constexpr int TX = TX_, TY = TY_, W = TX + 2, M = W * (TY + 2);
    static constexpr int THREADS = (M + 63) / 64 * 64;
    static constexpr int F = FLUID ? 1 : 0, H = THERMAL ? 1 : 0;
    static constexpr int GOFS = F * Q, LAG = GOFS + Q, PLANES = F * Q + H * (Q + 1);
};

// A node's results into LDS planes
template <int OFS, int M>
struct TileOut64 {
    double *t;
    int m;
    template <int q>
    __device__ void put(double v) const
    {
        t[(OFS + q) * M + m] = v;
    }
};

// The two steps of the tile whose first node is (x0, y0), through the block's
// LDS array t.
template <bool FLUID, bool THERMAL, bool NT, class T2>
__device__ __forceinline__ void step2_tile64(const KParams &P, const double *__restrict__ fin,
                                             const double *__restrict__ gin, double *__restrict__ fout,
                                             double *__restrict__ gout, const double *__restrict__ tl_in,
                                             double *__restrict__ tl_out, int x0, int y0, double *t)
{
    constexpr int M = T2::M, W = T2::W, TX = T2::TX, TY = T2::TY, G = T2::GOFS;
    const int NX = P.NX, NY = P.NY;
    const int w = NX - x0 < TX ? NX - x0 : TX;
    // first step (columns beyond the halo of a narrower last tile are never
    // read: skipped)
    if (const int m = threadIdx.x; m < M && m % W <= w + 1) {
        int x = x0 - 1 + m % W;  // in [-1, NX]
        x = x < 0 ? x + NX : (x >= NX ? x - NX : x);
        int y = (y0 - 1 + m / W) % NY;
        y = y < 0 ? y + NY : y;
        const uint32_t n = (uint32_t)y * NX + x;
        const Nbr b = make_nbr(x, y, 0, NX, NY, 1);
        const Pull<double, PULL_LINEAR> o(b, NX, NY);
        double f[Q], g[Q], Tlag = 0.0, T = 0.0;
        if constexpr (THERMAL) {
            Tlag = tl_in[n];
            pull_thermal64(P, b, make_planes(gin, P.S), o, Tlag, g);
        }
        if constexpr (FLUID) pull_fluid64(P, b, make_planes(fin, P.S), o, f);
        if constexpr (THERMAL) {
            T = m_sum(g);
            t[T2::LAG * M + m] = T;
        }
        collide64<FLUID, THERMAL, false>(P, b, f, g, Tlag, T, nullptr, n, TileOut64<0, M>{t, m}, TileOut64<G, M>{t, m});
    }
    __syncthreads();
    // second step
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int x = x0 + tx, y = y0 + ty;
    if (ty >= TY || y >= NY || tx >= w) return;
    const int at = (ty + 1) * W + tx + 1;
    const uint32_t n = (uint32_t)y * NX + x;
    const Nbr b = make_nbr(x, y, 0, NX, NY, 1);
    const Pull<double, PULL_LINEAR> o(b, NX, NY);
    double f[Q], g[Q], Tlag = 0.0, T = 0.0;
    if constexpr (THERMAL) {
        Tlag = t[T2::LAG * M + at];
        const double fac_top = 2.0 * (P.Tw_top - Tlag);
        const double fac_bot = 2.0 * (P.Tw_bot - Tlag);
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const bool cross = P.wall_t && crosses_wall<q>(b);
            const double v = t[(G + q) * M + (cross ? at : at - cxq(q) - cyq(q) * W)];
            if constexpr (cyq(q) > 0)
                g[q] = cross ? v + wq(q) * fac_bot : v;
            else if constexpr (cyq(q) < 0)
                g[q] = cross ? v + wq(q) * fac_top : v;
            else
                g[q] = v;
        });
        T = m_sum(g);
        tl_out[n] = T;
    }
    if constexpr (FLUID)
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const bool cross = P.wall_f && crosses_wall<q>(b);
            f[q] = cross ? t[invq(q) * M + at] : t[q * M + at - cxq(q) - cyq(q) * W];
        });
    collide64<FLUID, THERMAL, false>(P, b, f, g, Tlag, T, nullptr, n,
                                     PlaneOut<NT, PULL_LINEAR>{make_planes(FLUID ? fout : gout, P.S), o},
                                     PlaneOut<NT, PULL_LINEAR>{make_planes(THERMAL ? gout : fout, P.S), o});
}

template <bool FLUID, bool THERMAL, bool NT, class T2>
__global__ void __launch_bounds__(T2::THREADS) k_step2_fp64(KParams P, const double *__restrict__ fin,
                                                            const double *__restrict__ gin, double *__restrict__ fout,
                                                            double *__restrict__ gout,
                                                            const double *__restrict__ tl_in,
                                                            double *__restrict__ tl_out, int run)
{
    __shared__ double t[T2::PLANES * T2::M];
    const uint32_t lb = xcd_run(run, block_linear(), gridDim.x * gridDim.y), row = lb / gridDim.x;
    step2_tile64<FLUID, THERMAL, NT, T2>(P, fin, gin, fout, gout, tl_in, tl_out,
                                         (int)(lb - row * gridDim.x) * T2::TX, (int)row * T2::TY, t);
}

// Many 2-D lattices in one launch, two steps each or, where the slot says so,
// one (see k_step2_batch32).
template <bool FLUID, bool THERMAL, bool NT, class T2>
__global__ void __launch_bounds__(T2::THREADS) k_step2_batch64(const BatchEntry *__restrict__ tab,
                                                               const BatchSlot *__restrict__ slots, int nslots,
                                                               int run)
{
    __shared__ double t[T2::PLANES * T2::M];
    const uint32_t bt = xcd_run(run, blockIdx.x, gridDim.x);
    if (bt >= slots[nslots].tile0) return;
    int lo = 0, hi = nslots - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (slots[mid].tile0 <= bt)
            lo = mid;
        else
            hi = mid - 1;
    }
    const BatchSlot sl = slots[lo];
    const BatchEntry &E = tab[sl.entry & BATCH_ENTRY_MASK];
    const KParams &P = E.P;
    const int in = E.cur ^ (int)(sl.entry >> 31);
    const bool tp = (sl.entry & BATCH_LAG_PARITY) != 0;
    const double *fin = (const double *)E.f[in], *gin = (const double *)E.g[in];
    double *fout = (double *)E.f[in ^ 1], *gout = (double *)E.g[in ^ 1];
    double *tl_a = (double *)(tp ? E.tlag2 : E.tlag), *tl_b = (double *)(tp ? E.tlag : E.tlag2);
    const uint32_t tile = bt - sl.tile0, txs = ((uint32_t)P.NX + T2::TX - 1) / T2::TX;
    const int x0 = (int)(tile % txs) * T2::TX, y0 = (int)(tile / txs) * T2::TY;
    if (sl.entry & BATCH_SINGLE) {
        const int x = x0 + (int)threadIdx.x % T2::TX, y = y0 + (int)threadIdx.x / T2::TX;
        if ((int)threadIdx.x >= T2::TX * T2::TY || x >= P.NX || y >= P.NY) return;
        step_node64<false, FLUID, THERMAL, NT, false, true, PULL_LINEAR>(P, fin, gin, fout, gout, tl_a,
                                                                         (double *)E.taules, x, y, 0,
                                                                         (uint32_t)y * (uint32_t)P.NX + (uint32_t)x);
        return;
    }
    step2_tile64<FLUID, THERMAL, NT, T2>(P, fin, gin, fout, gout, tl_a, tl_b, x0, y0, t);
}

// Two steps per launch for 3-D lattices of few columns: a block owns R rows of
// all NX NZ columns (periodic within the block) and computes one row beside
// them in the first step, as k_step2_fp64 does with tiles.  Bound by the launch
// and by FP64 issue, so blocks are one wave per SIMD.  us per step, single ->
// this: channel 4x16x4 3.60 -> 2.90, 4x64x4 4.03 -> 2.95, 8x16x8 4.02 -> 2.99,
// 4x5000x4 8.3 -> 5.2; Rayleigh-Benard 8x16x4 5.2 -> 3.8, 8x64x8 5.4 -> 4.0.
// (One block with the whole lattice in LDS for any number of steps took 4.4 at
// 4x64x4: one CU's FP64 issue.)
constexpr int SLAB = 256;  // nodes of a block in the first step

// Rows of a block, 0 where this is not taken: at least six of them, or fewer in
// at most 32 blocks (3x300x21, two rows in 150 blocks: 5.4 against 4.4).
inline int slab_rows(const KParams &P)
{
    const int64_t R = SLAB / ((int64_t)P.NX * P.NZ) - 2;
    return R >= 6 || (R >= 2 && P.NY <= 32 * R) ? (int)R : 0;
}

template <bool FLUID, bool THERMAL>
__global__ void __launch_bounds__(SLAB) k_step2y_fp64(KParams P, const double *__restrict__ fin,
                                                      const double *__restrict__ gin, double *__restrict__ fout,
                                                      double *__restrict__ gout, const double *__restrict__ tl_in,
                                                      double *__restrict__ tl_out, int R)
{
    constexpr int G = FLUID ? Q : 0, LAG = G + Q;
    __shared__ double t[(G + (THERMAL ? Q + 1 : 0)) * SLAB];
    const int NX = P.NX, NY = P.NY, NZ = P.NZ, A = NX * NZ, m = threadIdx.x, r = m / A, c = m - r * A;
    const int x = c % NX, z = c / NX, y0 = (int)blockIdx.x * R;
    const bool act = r < R + 2;
    int y = (y0 - 1 + r) % NY;
    y = y < 0 ? y + NY : y;
    const uint32_t n = ((uint32_t)z * NY + y) * NX + x;
    const Nbr b = make_nbr(x, y, z, NX, NY, NZ);
    const Pull<double, PULL_LINEAR> o(b, NX, NY);
    double f[Q], g[Q], Tlag = 0.0, T = 0.0;
    if (act) {
        if constexpr (THERMAL) {
            Tlag = tl_in[n];
            pull_thermal64(P, b, make_planes(gin, P.S), o, Tlag, g);
        }
        if constexpr (FLUID) pull_fluid64(P, b, make_planes(fin, P.S), o, f);
        if constexpr (THERMAL) {
            T = m_sum(g);
            t[LAG * SLAB + m] = T;
        }
        collide64<FLUID, THERMAL, false>(P, b, f, g, Tlag, T, nullptr, n, TileOut64<0, SLAB>{t, m},
                                         TileOut64<G, SLAB>{t, m});
    }
    __syncthreads();
    if (r < 1 || r > R || y0 - 1 + r >= NY) return;
    // place in the block of the node at x - c_q
    auto src = [&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int xs = cxq(q) > 0 ? b.xm : (cxq(q) < 0 ? b.xp : x), zs = czq(q) > 0 ? b.zm : (czq(q) < 0 ? b.zp : z);
        return (r - cyq(q)) * A + zs * NX + xs;
    };
    if constexpr (THERMAL) {
        Tlag = t[LAG * SLAB + m];
        const double fac_top = 2.0 * (P.Tw_top - Tlag);
        const double fac_bot = 2.0 * (P.Tw_bot - Tlag);
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const bool cross = P.wall_t && crosses_wall<q>(b);
            const double v = t[(G + q) * SLAB + (cross ? m : src(qc))];
            if constexpr (cyq(q) > 0)
                g[q] = cross ? v + wq(q) * fac_bot : v;
            else if constexpr (cyq(q) < 0)
                g[q] = cross ? v + wq(q) * fac_top : v;
            else
                g[q] = v;
        });
        T = m_sum(g);
        tl_out[n] = T;
    }
    if constexpr (FLUID)
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const bool cross = P.wall_f && crosses_wall<q>(b);
            f[q] = cross ? t[invq(q) * SLAB + m] : t[q * SLAB + src(qc)];
        });
    collide64<FLUID, THERMAL, false>(P, b, f, g, Tlag, T, nullptr, n,
                                     PlaneOut<false, PULL_LINEAR>{make_planes(FLUID ? fout : gout, P.S), o},
                                     PlaneOut<false, PULL_LINEAR>{make_planes(THERMAL ? gout : fout, P.S), o});
}

// Velocity of the step at every node (the u[] that add_collision reads,
// fluid.c:1056-1080), for the finite-difference LES closure.
template <bool FIRST>
__global__ void __launch_bounds__(256) k_velocity64(KParams P, const double *__restrict__ fin,
                                                    const double *__restrict__ tlag)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y, z = blockIdx.z;
    if (x >= P.NX) return;
    const uint32_t n = ((uint32_t)z * P.NY + y) * P.NX + x;
    const size_t N = (size_t)P.N;
    const Nbr b = make_nbr(x, y, z, P.NX, P.NY, P.NZ);
    double f[Q];
    gather_fluid<FIRST>(P, b, fin, n, f);
    const double Tlag = P.thermal ? tlag[n] : 0.0;
    double rho, ux, uy, uz;
    fluid_velocity64(P, f, n, x, y, z, Tlag, rho, ux, uy, uz);
    double *vel = (double *)P.vel;
    vel[n] = ux;
    vel[N + n] = uy;
    vel[2 * N + n] = uz;
}

// Many lattices in one launch (see k_step_batch32).
template <bool FLUID, bool THERMAL, bool DENSE, bool NT, bool GEN, bool BUF>
__global__ void __launch_bounds__(256) k_step_batch64(const BatchEntry *__restrict__ tab,
                                                      const BatchSlot *__restrict__ slots, int nslots, int run)
{
    const uint32_t wt = __builtin_amdgcn_readfirstlane(xcd_run(run, blockIdx.x, gridDim.x) * BATCH_WAVES_PER_BLOCK +
                                                       threadIdx.x / BATCH_WAVE);
    if (wt >= slots[nslots].tile0) return;
    int lo = 0, hi = nslots - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (slots[mid].tile0 <= wt)
            lo = mid;
        else
            hi = mid - 1;
    }
    const BatchSlot sl = slots[lo];
    const BatchEntry &E = tab[sl.entry & BATCH_ENTRY_MASK];
    const KParams &P = E.P;
    const int in = E.cur ^ (int)(sl.entry >> 31);
    const double *fin = (const double *)E.f[in], *gin = (const double *)E.g[in];
    double *fout = (double *)E.f[in ^ 1], *gout = (double *)E.g[in ^ 1];
    double *tl = (double *)E.tlag, *tau = (double *)E.taules;
    // DENSE: wave tile t = nodes 64 t .. 64 t + 63 of the lattice, each lane
    // decoding its row; else tile t = up to 64 x of one row (row
    // coordinates wave-uniform), ceil(NX / 64) tiles per row
    const uint32_t t = wt - sl.tile0, lane = threadIdx.x % BATCH_WAVE;
    uint32_t n, x, y, z;
    if constexpr (DENSE) {
        n = t * BATCH_WAVE + lane;
        if (n >= (uint32_t)P.N) return;
        const uint32_t row = n / (uint32_t)P.NX;
        x = n - row * (uint32_t)P.NX;
        y = row % (uint32_t)P.NY;
        z = row / (uint32_t)P.NY;
    } else {
        const uint32_t xt = ((uint32_t)P.NX + BATCH_WAVE - 1) / BATCH_WAVE, row = t / xt;
        x = (t - row * xt) * BATCH_WAVE + lane;
        if (x >= (uint32_t)P.NX) return;
        y = row % (uint32_t)P.NY;
        z = row / (uint32_t)P.NY;
        n = row * (uint32_t)P.NX + x;
    }
    step_node64<false, FLUID, THERMAL, NT, GEN, BUF, DENSE ? PULL_LINEAR : PULL_ROW>(P, fin, gin, fout, gout, tl, tau, (int)x, (int)y, (int)z, n);
}

// Streaming of the last step + hydro_fields, without a new collision:
// produces the reference's p, g (records [N][19], as the host takes them),
// dens, u and t of the current step.  Any output may be null.
__global__ void __launch_bounds__(256) k_gather_fp64(KParams P, const double *__restrict__ fin,
                                                     const double *__restrict__ gin,
                                                     const double *__restrict__ tlag, double *__restrict__ fpost,
                                                     double *__restrict__ gpost, double *__restrict__ dens,
                                                     double *__restrict__ u, double *__restrict__ t)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= P.NX) return;
    const int y = blockIdx.y, z = blockIdx.z;
    const uint32_t n = ((uint32_t)z * P.NY + y) * P.NX + x;
    const Nbr b = make_nbr(x, y, z, P.NX, P.NY, P.NZ);
    double Tlag = 0.0;
    if (P.thermal) {
        double g[Q];
        Tlag = tlag[n];
        if (P.first)
            gather_thermal<true>(P, b, gin, n, Tlag, g);
        else
            gather_thermal<false>(P, b, gin, n, Tlag, g);
        if (gpost)
            for (int q = 0; q < Q; q++) gpost[(size_t)n * Q + q] = g[q];
        if (t) t[n] = m_sum(g);
    }
    if (P.fluid) {
        double f[Q];
        if (P.first)
            gather_fluid<true>(P, b, fin, n, f);
        else
            gather_fluid<false>(P, b, fin, n, f);
        if (fpost)
            for (int q = 0; q < Q; q++) fpost[(size_t)n * Q + q] = f[q];
        const double rho = m_sum(f);
        double ux, uy, uz;
        if (P.forced) {
            double F[3];
            force_at(P, P.hit_now, P.fb_now, P.f0n, n, x, y, z, Tlag, F);
            ux = m_x(f) / rho + 0.5 * 1.0 * F[0];
            uy = m_y(f) / rho + 0.5 * 1.0 * F[1];
            uz = m_z(f) / rho + 0.5 * 1.0 * F[2];
        } else {
            ux = m_x(f) / rho;
            uy = m_y(f) / rho;
            uz = m_z(f) / rho;
        }
        if (dens) dens[n] = rho;
        if (u) {
            u[3 * n] = ux;
            u[3 * n + 1] = uy;
            u[3 * n + 2] = uz;
        }
    }
}

static dim3 grid_of(const KParams &P, int bx) { return dim3((P.NX + bx - 1) / bx, P.NY, P.NZ); }
static int block_x(const KParams &P) { return P.NX >= 256 ? 256 : (P.NX >= 128 ? 128 : 64); }

void launch_step_fp64(const KParams &P, const double *fin, const double *gin, double *fout, double *gout,
                      double *tlag, double *taules, hipStream_t s)
{
    int bx = block_x(P);
    const bool dense = !P.first && dense_rows(P, 8);
    dim3 grid = grid_of(P, bx), block(bx);
    if (dense) {
        grid = dim3((unsigned)((P.N + 255) / 256));
        block = dim3(256);
    }
    const StepOrder o = step_order(state_bytes(P, 8), dense || P.NX % 16 == 0, CACHED_BYTES);
    // planes beyond the reach of buffer resources take the general instance
    const bool buf = planes_ok(P, 8), gen = P.hit || P.les || P.twoway || P.nozero || !buf;
    auto sets = [&](auto fl, auto th) {
        constexpr bool FL = decltype(fl)::value, TH = decltype(th)::value;
        if (P.first) {
            hipLaunchKernelGGL((k_step_fp64<true, FL, TH, false, false, true, false>), grid, block, 0, s, P, fin, gin,
                               fout, gout, tlag, taules, o.run);
            return;
        }
        with_bool(dense, [&](auto d) {
            with_bool(o.nts, [&](auto n) {
                constexpr bool D = decltype(d)::value, NT = decltype(n)::value;
                auto go = [&](auto g, auto bf) {
                    hipLaunchKernelGGL((k_step_fp64<false, FL, TH, D, NT, decltype(g)::value, decltype(bf)::value>),
                                       grid, block, 0, s, P, fin, gin, fout, gout, tlag, taules, o.run);
                };
                if (!gen)
                    go(std::false_type{}, std::true_type{});
                else if (buf)
                    go(std::true_type{}, std::true_type{});
                else
                    go(std::true_type{}, std::false_type{});
            });
        });
    };
    if (P.fluid && P.thermal)
        sets(std::true_type{}, std::true_type{});
    else if (P.fluid)
        sets(std::true_type{}, std::false_type{});
    else
        sets(std::false_type{}, std::true_type{});
}

// 2-D lattices whose rows leave much of their tiles idle: less than 60 % full,
// or a last tile of fewer than four columns in rows less than 80 % full (its
// lanes' loads and stores share no lines) while the launch is a few rounds of
// blocks.  Two steps pay for them only while one block per CU covers the lattice.  us per step, single -> two:
// Rayleigh-Benard 4x1000 5.1 -> 4.4, 16x1000 5.6 -> 3.8, 33x256 5.3 -> 5.4; with
// more tiles 1x30000 7.6 -> 57, 4x16000 7.7 -> 28, 16x4000 8.0 -> 8.9, 33x4000
// 14.5 -> 19.8, 97x1000 11.0 -> 12.9; channel 8x20000 11.7 -> 16.5; and full
// enough: 20x16000 -> 0.92 of single, 32x16000 56 -> 39, 40x4000 16.5 -> 16.9,
// 48x16000 99 -> 71, 65x16000 138 -> 109, 97x4000 36.7 -> 34.7, 100x1000 11.0 ->
// 10.5, 129x4000 -> 0.79.  Rows of one or two
// nodes take longer in two steps at any length (1x64 3.6 -> 5.3).
constexpr int64_t THIN_TILES = 256;
static bool thin2d(const KParams &P)
{
    const int64_t lanes = (P.NX + T2D_TX - 1) / T2D_TX * T2D_TX, last = P.NX - (lanes - T2D_TX);
    return (int64_t)P.NX * 10 < lanes * 6 ||
           (last < 4 && (int64_t)P.NX * 10 < lanes * 8 && batch2_tiles64(P.NX, P.NY) < 8 * THIN_TILES);
}

// tiles of a lattice that takes two steps only while its launch is that small
int64_t two_step_thin64(const KParams &P)
{
    return P.NZ == 1 && thin2d(P) ? batch2_tiles64(P.NX, P.NY) : 0;
}
bool two_step_thin_pays64(int64_t tiles) { return tiles <= THIN_TILES; }

// Two steps per launch (k_step2_fp64, k_step2y_fp64, k_step2z_fp64): lattices
// with the fluid whose planes buffer resources reach, without the general force
// paths.  2-D: see thin2d.
// Tiles: 32 x 8 with the temperature (141 KB of LDS), 64 x 8 without (135 KB).
using Tile64 = TileZ<true, true, 32, 8, true>;
using Tile64F = TileZ<true, false, 64, 8, true>;

static int64_t z_columns64(const KParams &P)
{
    const int tx = P.thermal ? Tile64::TX : Tile64F::TX, ty = P.thermal ? Tile64::TY : Tile64F::TY;
    return (int64_t)((P.NX + tx - 1) / tx) * ((P.NY + ty - 1) / ty);
}

// 3-D: where a launch's iterations (z_range) take less time than two single
// steps: 11.6 us each with the temperature (9.5 without), 9.1 (6.5) while the
// caches hold the state, against the nodes at 119 ps a step (57), 92 (49) in
// cache.  The rule leaves Rayleigh-Benard 64^3 (24 us per step against 27) and
// channels of 64^3 (13 against 19) and 78^3 (23 against 28) single, and takes
// channel 96^3 (46 against 39).
bool two_step_ok64(const KParams &P)
{
    if (!P.fluid || P.first || P.hit || P.les || P.twoway || P.nozero || !planes_ok(P, 8)) return false;
    if (P.NZ == 1) return !thin2d(P) || (P.NX >= 3 && two_step_thin_pays64(two_step_thin64(P)));
    if (slab_rows(P) > 0) return true;
    const bool cached = state_bytes(P, 8) <= CACHED_BYTES;
    const double t_iter = P.thermal ? (cached ? 9.1 : 11.6) : (cached ? 6.5 : 9.5);           // us
    const double t_node = P.thermal ? (cached ? 92e-6 : 119e-6) : (cached ? 49e-6 : 57e-6);  // us
    const int64_t columns = z_columns64(P);
    return (double)z_iterations(columns, P.NZ, z_range(columns, P.NZ)) * t_iter < 2.0 * (double)P.N * t_node;
}

bool two_step_slab64(const KParams &P) { return P.NZ > 1 && slab_rows(P) > 0; }

template <class TZ>
static void launch_z2_64(const KParams &P, const double *fin, const double *gin, double *fout, double *gout,
                         const double *tl_in, double *tl_out, hipStream_t s)
{
    const int zc = z_range(z_columns64(P), P.NZ);
    const dim3 grid((unsigned)((P.NX + TZ::TX - 1) / TZ::TX), (unsigned)((P.NY + TZ::TY - 1) / TZ::TY),
                    (unsigned)((P.NZ + zc - 1) / zc));
    constexpr bool FL = TZ::F == 1, TH = TZ::H == 1;
    with_bool(step_order(state_bytes(P, 8), P.NX % 8 == 0, 0).nts, [&](auto nt) {
        hipLaunchKernelGGL((k_step2z_fp64<FL, TH, decltype(nt)::value, TZ>), grid, dim3(TZ::THREADS), 0, s, P, fin,
                           gin, fout, gout, tl_in, tl_out, zc);
    });
}

template <class T2>
static void launch_2d_64(const KParams &P, const double *fin, const double *gin, double *fout, double *gout,
                         const double *tl_in, double *tl_out, hipStream_t s)
{
    const dim3 grid((unsigned)((P.NX + T2::TX - 1) / T2::TX), (unsigned)((P.NY + T2::TY - 1) / T2::TY));
    const StepOrder o = step_order(state_bytes(P, 8), P.NX % 16 == 0, RANGE_BYTES_2D);
    constexpr bool FL = T2::F == 1, TH = T2::H == 1;
    with_bool(o.nts, [&](auto nt) {
        hipLaunchKernelGGL((k_step2_fp64<FL, TH, decltype(nt)::value, T2>), grid, dim3(T2::THREADS), 0, s, P, fin, gin,
                           fout, gout, tl_in, tl_out, o.run);
    });
}

void launch_two_steps_fp64(const KParams &P, const double *fin, const double *gin, double *fout, double *gout,
                           const double *tl_in, double *tl_out, hipStream_t s)
{
    if (P.NZ == 1) {
        if (P.thermal)
            launch_2d_64<Tile2D<true, true, T2D_TX, T2D_TY>>(P, fin, gin, fout, gout, tl_in, tl_out, s);
        else
            launch_2d_64<Tile2D<true, false, T2D_TX, T2D_TY>>(P, fin, gin, fout, gout, tl_in, tl_out, s);
        return;
    }
    if (const int R = slab_rows(P); R > 0) {
        const dim3 grid((unsigned)((P.NY + R - 1) / R));
        if (P.thermal)
            hipLaunchKernelGGL((k_step2y_fp64<true, true>), grid, dim3(SLAB), 0, s, P, fin, gin, fout, gout, tl_in,
                               tl_out, R);
        else
            hipLaunchKernelGGL((k_step2y_fp64<true, false>), grid, dim3(SLAB), 0, s, P, fin, gin, fout, gout, tl_in,
                               tl_out, R);
        return;
    }
    if (P.thermal)
        launch_z2_64<Tile64>(P, fin, gin, fout, gout, tl_in, tl_out, s);
    else
        launch_z2_64<Tile64F>(P, fin, gin, fout, gout, tl_in, tl_out, s);
}

void launch_velocity_fp64(const KParams &P, const double *fin, const double *tlag, hipStream_t s)
{
    int bx = block_x(P);
    dim3 grid = grid_of(P, bx);
    if (P.first)
        hipLaunchKernelGGL(k_velocity64<true>, grid, dim3(bx), 0, s, P, fin, tlag);
    else
        hipLaunchKernelGGL(k_velocity64<false>, grid, dim3(bx), 0, s, P, fin, tlag);
}

void launch_batch_fp64(const BatchEntry *tab, const BatchSlot *slots, int nslots, int64_t nblocks, int kind,
                       bool dense, bool gen, bool buf, StepOrder o, hipStream_t s)
{
    dim3 grid((unsigned)nblocks), block(256);
    gen = gen || !buf;
    auto sets = [&](auto fl, auto th) {
        constexpr bool FL = decltype(fl)::value, TH = decltype(th)::value;
        with_bool(dense, [&](auto d) {
            with_bool(o.nts, [&](auto n) {
                constexpr bool D = decltype(d)::value, NT = decltype(n)::value;
                auto go = [&](auto g, auto bf) {
                    hipLaunchKernelGGL((k_step_batch64<FL, TH, D, NT, decltype(g)::value, decltype(bf)::value>), grid,
                                       block, 0, s, tab, slots, nslots, o.run);
                };
                if (!gen)
                    go(std::false_type{}, std::true_type{});
                else if (buf)
                    go(std::true_type{}, std::true_type{});
                else
                    go(std::true_type{}, std::false_type{});
            });
        });
    };
    if (kind == BATCH_FLUID_THERMAL)
        sets(std::true_type{}, std::true_type{});
    else if (kind == BATCH_FLUID)
        sets(std::true_type{}, std::false_type{});
    else
        sets(std::false_type{}, std::true_type{});
}

int64_t batch2_tiles64(int NX, int NY)
{
    return (int64_t)((NX + T2D_TX - 1) / T2D_TX) * ((NY + T2D_TY - 1) / T2D_TY);
}

void launch_batch2_fp64(const BatchEntry *tab, const BatchSlot *slots, int nslots, int64_t nblocks, int kind,
                        StepOrder o, hipStream_t s)
{
    auto go = [&](auto th) {
        constexpr bool TH = decltype(th)::value;
        using T2 = Tile2D<true, TH, T2D_TX, T2D_TY>;
        with_bool(o.nts, [&](auto nt) {
            hipLaunchKernelGGL((k_step2_batch64<true, TH, decltype(nt)::value, T2>), dim3((unsigned)nblocks),
                               dim3(T2::THREADS), 0, s, tab, slots, nslots, o.run);
        });
    };
    if (kind == BATCH_FLUID_THERMAL)
        go(std::true_type{});
    else
        go(std::false_type{});
}

// LB_FLUID_FORCING_NOZEROMODE (forcing.c:1123-1152): sums over all nodes of
// the built force (no particle feedback) of the previous step, F(Tlag) with
// the previous HIT table, and of this step, F(T) with T gathered as the step
// kernel gathers it (STEP), or of the last step alone, F(Tlag) with the
// current table (the hydro-fields gather).  Fixed grid and a tree per block:
// the partial sums are the same on every run.
constexpr int FM_THREADS = 256, FM_BLOCKS = 512;

template <bool STEP, bool FIRST>
__global__ void __launch_bounds__(FM_THREADS) k_force_sum64(KParams P, const double *__restrict__ gin,
                                                            const double *__restrict__ tlag, double *__restrict__ part)
{
    P.twoway = 0;
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const int64_t N = P.N, stride = (int64_t)gridDim.x * FM_THREADS;
    for (int64_t i = (int64_t)blockIdx.x * FM_THREADS + threadIdx.x; i < N; i += stride) {
        const uint32_t n = (uint32_t)i;
        const int x = (int)(i % P.NX), y = (int)((i / P.NX) % P.NY), z = (int)(i / ((int64_t)P.NX * P.NY));
        const double Tlag = P.thermal ? tlag[n] : 0.0;
        double F[3];
        if constexpr (STEP) {
            force_at(P, P.hit_prev, nullptr, nullptr, n, x, y, z, Tlag, F);
            for (int c = 0; c < 3; c++) acc[c] += F[c];
            double T = 0.0;
            if (P.thermal && P.buoy) {
                double g[Q];
                gather_thermal<FIRST>(P, make_nbr(x, y, z, P.NX, P.NY, P.NZ), gin, n, Tlag, g);
                T = m_sum(g);
            }
            force_at(P, P.hit_now, nullptr, nullptr, n, x, y, z, T, F);
        } else {
            force_at(P, P.hit_now, nullptr, nullptr, n, x, y, z, Tlag, F);
        }
        for (int c = 0; c < 3; c++) acc[3 + c] += F[c];
    }
    __shared__ double red[6][FM_THREADS];
    for (int c = 0; c < 6; c++) red[c][threadIdx.x] = acc[c];
    __syncthreads();
    for (int w = FM_THREADS / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int c = 0; c < 6; c++) red[c][threadIdx.x] += red[c][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 6) part[(size_t)blockIdx.x * 6 + threadIdx.x] = red[threadIdx.x][0];
}

// Block sums in block order, times 1/(NX NY NZ) as forcing.c:1140 forms it.
__global__ void k_force_mean64(int nblocks, double NX, double NY, double NZ, const double *__restrict__ part,
                               double *__restrict__ f0)
{
    const int c = threadIdx.x;
    if (c >= 6) return;
    double s = 0.0;
    for (int b = 0; b < nblocks; b++) s += part[(size_t)b * 6 + c];
    const double norm = 1.0 / (NX * NY * NZ);
    f0[c] = s * norm;
}

// f0[0..2]: mean force of the previous step, f0[3..5]: of this step (STEP);
// without STEP only f0[3..5] (the last step's).  part: FM_BLOCKS * 6 doubles.
void launch_force_mean64(const KParams &P, bool step, const double *gin, const double *tlag, double *part, double *f0,
                         hipStream_t s)
{
    const int64_t need = (P.N + FM_THREADS - 1) / FM_THREADS;
    const int nb = (int)(need < FM_BLOCKS ? need : FM_BLOCKS);
    if (!step)
        hipLaunchKernelGGL((k_force_sum64<false, false>), dim3(nb), dim3(FM_THREADS), 0, s, P, gin, tlag, part);
    else if (P.first)
        hipLaunchKernelGGL((k_force_sum64<true, true>), dim3(nb), dim3(FM_THREADS), 0, s, P, gin, tlag, part);
    else
        hipLaunchKernelGGL((k_force_sum64<true, false>), dim3(nb), dim3(FM_THREADS), 0, s, P, gin, tlag, part);
    hipLaunchKernelGGL(k_force_mean64, dim3(1), dim3(64), 0, s, nb, (double)P.NX, (double)P.NY, (double)P.NZ, part, f0);
}

void launch_gather_fp64(const KParams &P, const double *fin, const double *gin, const double *tlag, double *fpost,
                        double *gpost, double *dens, double *u, double *t, hipStream_t s)
{
    int bx = block_x(P);
    hipLaunchKernelGGL(k_gather_fp64, grid_of(P, bx), dim3(bx), 0, s, P, fin, gin, tlag, fpost, gpost, dens, u, t);
}

}  // namespace ch4g
