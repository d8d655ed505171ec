// Initialisation, population load, and the FP64 reductions of dump_averages.
// Compiled with -ffp-contract=off: the FP64 init arithmetic (g = w t,
// p = w, t = sum g) must equal the reference's bit for bit.
#include "ch4g_internal.h"

namespace ch4g {

__device__ __forceinline__ int wrapc(int a, int L) { return a < 0 ? a + L : (a >= L ? a - L : a); }

__device__ __forceinline__ double msum19(const double *p)
{
    return p[0] + p[1] + p[2] + p[3] + p[4] + p[5] + p[6] + p[7] + p[8] + p[9] + p[10] + p[11] + p[12] + p[13] +
           p[14] + p[15] + p[16] + p[17] + p[18];
}

// initial_conditions on the device from a per-row fluid profile prow[y][19]
// and a temperature field t0[n] built on the host (initial_conditions.c:45,
// :72-84, :256-279, :303-308, :421-424, :486-487); tlag <- sum g (the t of
// the first hydro_fields call, main.c:29-31).
template <typename R>
__global__ void k_init(KParams P, const double *__restrict__ prow, const double *__restrict__ t0,
                       R *__restrict__ f, R *__restrict__ g, R *__restrict__ tlag, int dev)
{
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= P.N) return;
    const int y = (int)((n / P.NX) % P.NY);
    // FP32-deviation: subtract the per-row base state (rho_b, T_b)
    const double rb = dev ? P.row64[2 * y] : 0.0, tb = dev ? P.row64[2 * y + 1] : 0.0;
    if (P.fluid) {
        for (int q = 0; q < Q; q++) {
            double v = prow[y * Q + q];
            f[q * P.S + n] = dev ? (R)(v - wq(q) * rb) : (R)v;
        }
    }
    if (P.thermal) {
        double gq[Q];
        double t = t0[n];
        for (int q = 0; q < Q; q++) gq[q] = wq(q) * t;
        for (int q = 0; q < Q; q++) g[q * P.S + n] = dev ? (R)(gq[q] - wq(q) * tb) : (R)gq[q];
        double T = msum19(gq);
        tlag[n] = dev ? (R)(T - tb) : (R)T;
    }
}

// Load populations from the host's FP64 records [N][19] (restart), tlag <-
// sum g.  A wave reads 64 consecutive records: their lines stay in the L1
// over the 19 strided reads.
template <typename R>
__global__ void k_load(KParams P, const double *__restrict__ fs, const double *__restrict__ gs, R *__restrict__ f,
                       R *__restrict__ g, R *__restrict__ tlag, int dev)
{
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= P.N) return;
    const int y = (int)((n / P.NX) % P.NY);
    const double rb = dev ? P.row64[2 * y] : 0.0, tb = dev ? P.row64[2 * y + 1] : 0.0;
    if (P.fluid && fs)
        for (int q = 0; q < Q; q++) {
            double v = fs[n * Q + q];
            f[q * P.S + n] = dev ? (R)(v - wq(q) * rb) : (R)v;
        }
    if (P.thermal && gs) {
        double gq[Q];
        for (int q = 0; q < Q; q++) gq[q] = gs[n * Q + q];
        for (int q = 0; q < Q; q++) g[q * P.S + n] = dev ? (R)(gq[q] - wq(q) * tb) : (R)gq[q];
        double T = msum19(gq);
        tlag[n] = dev ? (R)(T - tb) : (R)T;
    }
}

void launch_init(const KParams &P, const double *prow, const double *t0, void *f, void *g, void *tlag, int dev,
                 hipStream_t s)
{
    int64_t nb = (P.N + 255) / 256;
    if (dev)
        hipLaunchKernelGGL(k_init<float>, dim3((unsigned)nb), dim3(256), 0, s, P, prow, t0, (float *)f, (float *)g,
                           (float *)tlag, 1);
    else
        hipLaunchKernelGGL(k_init<double>, dim3((unsigned)nb), dim3(256), 0, s, P, prow, t0, (double *)f,
                           (double *)g, (double *)tlag, 0);
}

void launch_load(const KParams &P, const double *fs, const double *gs, void *f, void *g, void *tlag, int dev,
                 hipStream_t s)
{
    int64_t nb = (P.N + 255) / 256;
    if (dev)
        hipLaunchKernelGGL(k_load<float>, dim3((unsigned)nb), dim3(256), 0, s, P, fs, gs, (float *)f, (float *)g,
                           (float *)tlag, 1);
    else
        hipLaunchKernelGGL(k_load<double>, dim3((unsigned)nb), dim3(256), 0, s, P, fs, gs, (double *)f,
                           (double *)g, (double *)tlag, 0);
}

// ---------------------------------------------------------------------------
// dump_averages (output.c:183-491): per-node FP64 contributions, centred
// differences with periodic wrap, one-sided second order at y walls
// (gradients.c:78-499, :505-626), summed in a fixed order.  Output order =
// ch4g_output.
//
// Every node's terms need the fields of seven nodes (29 doubles of which 5
// are new), so a wave takes 64 x of a row and marches: along y for the sums
// over x-y planes (k_plane_sums: averages, z ruler), along z for those over
// the other planes (k_column_sums: x and y rulers), with the node and its two
// neighbours along the march in registers and the sums in registers over the
// whole march.  256^3, us, one node per thread and one LDS tree per term ->
// this: averages 630 -> 280 (0.67 GB of fields), final sum 616 -> 8; rulers,
// one block per plane before, x 3480, y 744, z 660 -> 670 together.  Small
// lattices: 32 -> 10 for the averages.  Lattices narrower than a wave put several
// rows into one for the plane sums (us an averages call, one row a wave -> this:
// 1x1000x1000 1950 -> 1330, 8x256x256 170 -> 137, 3x300x21 74 -> 48).

constexpr int RED_THREADS = 256, RED_WAVES = RED_THREADS / 64;
constexpr int NTERM = 25;  // ch4g_output without lb, which is formed from the sums

// work of one block: unit = (z plane, part of it); a part is RED_WAVES waves,
// each lx x of 64 / lx groups of `rows` consecutive rows (lx: 64 or, for
// narrower lattices, the power of two that holds a row)
struct PlaneWork {
    int lx, nxt, rows, parts;
    int64_t units;
};

static PlaneWork plane_work(const KParams &P)
{
    PlaneWork w;
    w.lx = 64;
    while (w.lx / 2 >= P.NX) w.lx /= 2;
    w.nxt = (P.NX + w.lx - 1) / w.lx;
    const int groups = 64 / w.lx;
    // rows per lane: up to 16 (the two rows next to a march are read again),
    // fewer where that would leave less than 4 waves per SIMD
    const int64_t waves = (int64_t)w.nxt * ((P.NY + groups - 1) / groups) * P.NZ;
    const int64_t r = waves / 4096;
    w.rows = (int)(r < 1 ? 1 : (r > 16 ? 16 : r));
    const int64_t tasks = (int64_t)w.nxt * ((P.NY + groups * w.rows - 1) / (groups * w.rows));
    w.parts = (int)((tasks + RED_WAVES - 1) / RED_WAVES);
    w.units = (int64_t)w.parts * P.NZ;
    return w;
}

// blocks of the averages' sum, each over every gridDim-th unit
int reduce_blocks(const KParams &P)
{
    const int64_t nb = plane_work(P).units;
    return (int)(nb < 2048 ? nb : 2048);
}

// the fields of one node (0 for a set the lattice lacks)
struct FieldNode {
    double u[3], t;
};

struct Fields {
    const double *__restrict__ dens, *__restrict__ u, *__restrict__ t;
    int fluid, thermal;
    __device__ __forceinline__ FieldNode at(int64_t n) const
    {
        FieldNode v;
        v.u[0] = fluid ? u[3 * n] : 0.0;
        v.u[1] = fluid ? u[3 * n + 1] : 0.0;
        v.u[2] = fluid ? u[3 * n + 2] : 0.0;
        v.t = thermal ? t[n] : 0.0;
        return v;
    }
};

__device__ __forceinline__ FieldNode centred(const FieldNode &p, const FieldNode &m, bool flat)
{
    FieldNode g;
    for (int c = 0; c < 3; c++) g.u[c] = flat ? 0.0 : (p.u[c] - m.u[c]) / 2.0;
    g.t = (p.t - m.t) / 2.0;
    return g;
}

// y derivative at row y of column (x, z) from the rows next to it
__device__ __forceinline__ FieldNode dy_at(const KParams &P, const Fields &F, const FieldNode &c, const FieldNode &m,
                                           const FieldNode &p, int64_t n, int y)
{
    FieldNode g = centred(p, m, P.NY == 1);
    if ((P.wall_f || P.wall_t) && P.NY >= 3 && (y == 0 || y == P.NY - 1)) {
        const bool lo = y == 0;
        const FieldNode e = F.at(lo ? n + 2 * (int64_t)P.NX : n - 2 * (int64_t)P.NX);
        if (P.wall_f)
            for (int k = 0; k < 3; k++)
                g.u[k] = lo ? -1.5 * c.u[k] + 2.0 * p.u[k] - 0.5 * e.u[k] : 1.5 * c.u[k] - 2.0 * m.u[k] + 0.5 * e.u[k];
        if (P.wall_t) g.t = lo ? -1.5 * c.t + 2.0 * p.t - 0.5 * e.t : 1.5 * c.t - 2.0 * m.t + 0.5 * e.t;
    }
    return g;
}

// Per-node terms of dump_averages (output.c:183-491) added into a[] in the
// order of ch4g_output, from the node's fields and their derivatives.
__device__ __forceinline__ void add_terms(const KParams &P, double nu, double kappa, double dens, const FieldNode &c,
                                          const FieldNode &dx, const FieldNode &dy, const FieldNode &dz, int x, int y,
                                          int z, double a[NTERM])
{
    const double ux = c.u[0], uy = c.u[1], uz = c.u[2];
    if (P.fluid) {
        a[0] += (double)x + 0.5;
        a[1] += (double)y + 0.5;
        a[2] += (double)z + 0.5;
        a[3] += ux;
        a[4] += uy;
        a[5] += uz;
        a[6] += ux * ux;
        a[7] += uy * uy;
        a[8] += uz * uz;
        a[9] += dens;
        a[10] += 0.5 * (ux * ux + uy * uy + uz * uz);
        a[12] += dens * dens;
        double e = 0.0;
        for (int i = 0; i < 3; i++) {
            const double G[3] = {dx.u[i], dy.u[i], dz.u[i]}, H[3] = {i == 0 ? dx.u[0] : i == 1 ? dy.u[0] : dz.u[0],
                                                                     i == 0 ? dx.u[1] : i == 1 ? dy.u[1] : dz.u[1],
                                                                     i == 0 ? dx.u[2] : i == 1 ? dy.u[2] : dz.u[2]};
            for (int d = 0; d < 3; d++) {
                const double s = G[d] + H[d];
                e += s * s;
            }
        }
        a[11] += e * 0.5 * nu;
    }
    if (P.thermal) {
        const double t = c.t, gx = dx.t, gy = dy.t, gz = dz.t;
        a[13] += t;
        a[14] += t * t;
        a[15] += kappa * (gx * gx + gy * gy + gz * gz);
        a[16] += gx;
        a[17] += gy;
        a[18] += gz;
        a[19] += ux * t;
        a[20] += uy * t;
        a[21] += uz * t;
        a[22] += -kappa * gx + ux * t;
        a[23] += -kappa * gy + uy * t;
        a[24] += -kappa * gz + uz * t;
    }
}

// sum over the 64 lanes, the same in every lane
__device__ __forceinline__ double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sums over parts of x-y planes.  PER_UNIT: out[unit] (z ruler); else
// out[block], over every gridDim-th unit (averages).
template <bool PER_UNIT>
__global__ void __launch_bounds__(RED_THREADS) k_plane_sums(KParams P, Fields F, double nu, double kappa, PlaneWork w,
                                                            double *__restrict__ out)
{
    const int NX = P.NX, NY = P.NY, NZ = P.NZ;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    double a[NTERM];
    for (int k = 0; k < NTERM; k++) a[k] = 0.0;
    const uint32_t first = xcd_block(blockIdx.x, gridDim.x);
    for (int64_t unit = first; unit < w.units; unit += gridDim.x) {
        const int z = (int)(unit / w.parts), task = (int)(unit - (int64_t)z * w.parts) * RED_WAVES + wave;
        const int x = task % w.nxt * w.lx + lane % w.lx;
        const int y0 = (task / w.nxt * (64 / w.lx) + lane / w.lx) * w.rows, y1 = min(y0 + w.rows, NY);
        if (x < NX && y0 < NY) {
            const int64_t plane = (int64_t)z * NY * NX;
            const int64_t dzp = (int64_t)(wrapc(z + 1, NZ) - z) * NY * NX, dzm = (int64_t)(wrapc(z - 1, NZ) - z) * NY * NX;
            const int dxp = wrapc(x + 1, NX) - x, dxm = wrapc(x - 1, NX) - x;
            FieldNode m = F.at(plane + (int64_t)wrapc(y0 - 1, NY) * NX + x), c = F.at(plane + (int64_t)y0 * NX + x);
            for (int y = y0; y < y1; y++) {
                const int64_t n = plane + (int64_t)y * NX + x;
                const FieldNode p = F.at(plane + (int64_t)wrapc(y + 1, NY) * NX + x);
                const FieldNode dx = centred(F.at(n + dxp), F.at(n + dxm), NX == 1);
                const FieldNode dz = centred(F.at(n + dzp), F.at(n + dzm), NZ == 1);
                add_terms(P, nu, kappa, P.fluid ? F.dens[n] : 0.0, c, dx, dy_at(P, F, c, m, p, n, y), dz, x, y, z, a);
                m = c;
                c = p;
            }
        }
        if constexpr (PER_UNIT) break;  // one unit per block
    }
    __shared__ double sh[RED_WAVES][NTERM];
    for (int k = 0; k < NTERM; k++) {
        const double v = wave_sum(a[k]);
        if (lane == 0) sh[wave][k] = v;
    }
    __syncthreads();
    if (threadIdx.x < NOUT) {
        double s = 0.0;
        if (threadIdx.x < NTERM)
            for (int i = 0; i < RED_WAVES; i++) s += sh[i][threadIdx.x];
        out[(int64_t)first * NOUT + threadIdx.x] = s;
    }
}

// columns of the x and y rulers: a block is RED_WAVES waves on consecutive
// groups of `rows` rows, 64 x and zc planes
struct ColumnWork {
    int nxt, rows, nyb, zc, nzc;
};

static ColumnWork column_work(const KParams &P)
{
    ColumnWork w;
    w.nxt = (P.NX + 63) / 64;
    w.zc = P.NZ < 32 ? P.NZ : 32;
    w.nzc = (P.NZ + w.zc - 1) / w.zc;
    const int64_t blocks = (int64_t)w.nxt * ((P.NY + RED_WAVES - 1) / RED_WAVES) * w.nzc, r = blocks / 2048;
    w.rows = (int)(r < 1 ? 1 : (r > 8 ? 8 : r));
    w.nyb = (P.NY + RED_WAVES * w.rows - 1) / (RED_WAVES * w.rows);
    return w;
}

// Sums along z, then over the rows of a block (px[yb * nzc + zi][x]) and over
// the 64 x of a wave (py[xt * nzc + zi][y]).
__global__ void __launch_bounds__(RED_THREADS) k_column_sums(KParams P, Fields F, double nu, double kappa,
                                                             ColumnWork w, double *__restrict__ px,
                                                             double *__restrict__ py)
{
    const int NX = P.NX, NY = P.NY, NZ = P.NZ;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
    const int xt = lb % w.nxt, yb = lb / w.nxt % w.nyb, zi = lb / w.nxt / w.nyb;
    const int x = xt * 64 + lane, z0 = zi * w.zc, z1 = min(z0 + w.zc, NZ);
    const int64_t plane = (int64_t)NX * NY;
    double cx[NTERM];
    for (int k = 0; k < NTERM; k++) cx[k] = 0.0;
    for (int r = 0; r < w.rows; r++) {
        const int y = (yb * RED_WAVES + wave) * w.rows + r;
        if (y >= NY) break;
        double a[NTERM];
        for (int k = 0; k < NTERM; k++) a[k] = 0.0;
        if (x < NX) {
            const int64_t row = (int64_t)y * NX + x;
            const int dxp = wrapc(x + 1, NX) - x, dxm = wrapc(x - 1, NX) - x;
            const int64_t dyp = (int64_t)(wrapc(y + 1, NY) - y) * NX, dym = (int64_t)(wrapc(y - 1, NY) - y) * NX;
            FieldNode m = F.at(row + wrapc(z0 - 1, NZ) * plane), c = F.at(row + z0 * plane);
            for (int z = z0; z < z1; z++) {
                const int64_t n = row + z * plane;
                const FieldNode p = F.at(row + wrapc(z + 1, NZ) * plane);
                const FieldNode dx = centred(F.at(n + dxp), F.at(n + dxm), NX == 1);
                const FieldNode dy = dy_at(P, F, c, F.at(n + dym), F.at(n + dyp), n, y);
                add_terms(P, nu, kappa, P.fluid ? F.dens[n] : 0.0, c, dx, dy, centred(p, m, NZ == 1), x, y, z, a);
                m = c;
                c = p;
            }
        }
        double *o = py + ((int64_t)(xt * w.nzc + zi) * NY + y) * NOUT;
        for (int k = 0; k < NTERM; k++) {
            cx[k] += a[k];
            const double v = wave_sum(a[k]);
            if (lane == 0) o[k] = v;
        }
        if (lane == 0) o[NTERM] = 0.0;
    }
    // the block's waves, term by term
    __shared__ double sh[RED_WAVES][64];
    for (int k = 0; k < NTERM; k++) {
        sh[wave][lane] = cx[k];
        __syncthreads();
        if (wave == 0 && x < NX) {
            double s = 0.0;
            for (int i = 0; i < RED_WAVES; i++) s += sh[i][lane];
            px[((int64_t)(yb * w.nzc + zi) * NX + x) * NOUT + k] = s;
        }
        __syncthreads();
    }
    if (wave == 0 && x < NX) px[((int64_t)(yb * w.nzc + zi) * NX + x) * NOUT + NTERM] = 0.0;
}

// out[p] = sum of the `count` records in[p * pstride + i * istride] (records
// of NOUT doubles; 32 lanes a record, 32 records at a time, then a tree)
constexpr int SUM_ROWS = 32;
__global__ void __launch_bounds__(32 * SUM_ROWS) k_sum_records(const double *__restrict__ in, int64_t count,
                                                               int64_t istride, int64_t pstride,
                                                               double *__restrict__ out)
{
    const int k = threadIdx.x % 32, r = threadIdx.x / 32;
    const double *p = in + (int64_t)blockIdx.x * pstride * NOUT;
    double s = 0.0;
    if (k < NOUT) {
        // eight loads in flight: one at a time, 2048 records take 30 us
        int64_t i = r;
        for (; i + 7 * SUM_ROWS < count; i += 8 * SUM_ROWS) {
            double v[8];
            for (int j = 0; j < 8; j++) v[j] = p[(i + j * SUM_ROWS) * istride * NOUT + k];
            for (int j = 0; j < 8; j++) s += v[j];
        }
        for (; i < count; i += SUM_ROWS) s += p[i * istride * NOUT + k];
    }
    __shared__ double sh[SUM_ROWS][32];
    sh[r][k] = s;
    for (int h = SUM_ROWS / 2; h > 0; h >>= 1) {
        __syncthreads();
        if (r < h) sh[r][k] += sh[r + h][k];
    }
    if (r == 0 && k < NOUT) out[(int64_t)blockIdx.x * NOUT + k] = sh[0][k];
}

size_t ruler_scratch_doubles(const KParams &P)
{
    const ColumnWork c = column_work(P);
    const int64_t planes = plane_work(P).units;
    const int64_t cols = (int64_t)c.nzc * ((int64_t)c.nyb * P.NX + (int64_t)c.nxt * P.NY);
    return (size_t)(planes > cols ? planes : cols) * NOUT;
}

void launch_rulers(const KParams &P, const double *dens, const double *u, const double *t, double nu, double kappa,
                   double *scratch, double *rx, double *ry, double *rz, hipStream_t s)
{
    const Fields F{dens, u, t, P.fluid, P.thermal};
    const dim3 sum(32 * SUM_ROWS);
    if (rz) {
        const PlaneWork w = plane_work(P);
        hipLaunchKernelGGL(k_plane_sums<true>, dim3((unsigned)w.units), dim3(RED_THREADS), 0, s, P, F, nu, kappa, w,
                           scratch);
        hipLaunchKernelGGL(k_sum_records, dim3(P.NZ), sum, 0, s, scratch, w.parts, 1, w.parts, rz);
    }
    if (rx || ry) {
        const ColumnWork w = column_work(P);
        double *px = scratch, *py = scratch + (int64_t)w.nyb * w.nzc * P.NX * NOUT;
        hipLaunchKernelGGL(k_column_sums, dim3((unsigned)w.nxt * w.nyb * w.nzc), dim3(RED_THREADS), 0, s, P, F, nu,
                           kappa, w, px, py);
        if (rx) hipLaunchKernelGGL(k_sum_records, dim3(P.NX), sum, 0, s, px, (int64_t)w.nyb * w.nzc, P.NX, 1, rx);
        if (ry) hipLaunchKernelGGL(k_sum_records, dim3(P.NY), sum, 0, s, py, (int64_t)w.nxt * w.nzc, P.NY, 1, ry);
    }
}

void launch_averages(const KParams &P, const double *dens, const double *u, const double *t, double nu, double kappa,
                     double *partials, double *result, hipStream_t s)
{
    const int nb = reduce_blocks(P);
    hipLaunchKernelGGL(k_plane_sums<false>, dim3(nb), dim3(RED_THREADS), 0, s, P, Fields{dens, u, t, P.fluid, P.thermal},
                       nu, kappa, plane_work(P), partials);
    hipLaunchKernelGGL(k_sum_records, dim3(1), dim3(32 * SUM_ROWS), 0, s, partials, nb, 1, 0, result);
}

}  // namespace ch4g
