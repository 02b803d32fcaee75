// k_mls.hip -- MLS transport of the FP64 formulation on gfx950: the normal
// equations assembled and solved every step, per particle and velocity node
// (k_transport3d, k_transport2d) or, in 3-D, once per node for all particles
// whose stencils are congruent (k_stencil_coef, k_apply_runs).
//
// Per particle: one thread per (particle, velocity node), coalesced over the
// node index; a workgroup covers 256 nodes of one particle and stages that
// particle's neighbour offsets in LDS (every lane reads the same entry: an LDS
// broadcast). Interior and boundary particles come from compact lists, each
// with its compile-time basis size, instead of sweeping the whole grid twice
// with early exits as the reference does (CudaBackend.cu:1667-1677).
//
// What bounds that is the count of FP64 instructions per neighbour, so the
// assembly keeps the distinct sums only. A = sum w phi phi^T of the quadratic
// basis has 55 entries in its upper triangle but 35 distinct monomials
// sum w x^a y^b z^c (15 of 21 in 2-D); they are built as a chain of products
// (w, wx, wxx, ...), which the right-hand side shares. Offsets are scaled by
// 1/h once per particle, so no neighbour needs a division: 73 FP64
// instructions per neighbour and node instead of about 140 with four
// divisions and the full triangle. 2-D, 100^2 / Nv 44, linear: 1.26 -> 0.62 ms.
#include "ab_device.hpp"
#include "ab_internal.hpp"
#include "ab_mls.hpp"

#include <algorithm>

namespace ab {

namespace {

// Workgroups that fill 256 CUs with the register-heaviest transport kernel
// (three waves per SIMD: three workgroups per CU), twice over.
constexpr int kFillBlocks = 256 * 6;

// One item (particle i, 256 nodes) of kCopyGt + kTransportNode3DT<P, BND> (Solver/CudaBackend.cu:191-197, 699-869).
// DIAG: the degeneracy and overshoot flags of the step statistics, and the
// optional clamp, which need the neighbours' range at every node; without
// them nothing reads the range and it is not formed.
// 40^3 / Nv 10, quadratic: interior and boundary launch together 25.5 -> 13.6
// ms with the distinct sums (64,000 x 1,000 nodes, 78 Tflop/s FP64 vector rate).
template <int P, bool BND, bool DIAG>
__device__ __forceinline__ void transport3d_item(const DevCloud &c, const double *__restrict__ g,
                                                 double *__restrict__ gt, double dt, double h,
                                                 double tol, int clamp, int *mlsflag,
                                                 double *mlsovr, int i, int chunk,
                                                 double (&se)[AB_MAX_NEIGH][4],
                                                 int (&sj)[AB_MAX_NEIGH])
{
    const int lin = chunk * kBlock + threadIdx.x;
    const int nn = c.nneigh[i];
    const double ih = 1.0 / h;
    const double xi = c.x[i], yi = c.y[i], zi = c.z[i];
    __syncthreads();                         // the last item's readers are done
    for (int t = threadIdx.x; t < nn; t += kBlock)
    {
        const int j = c.neigh[(size_t)i * AB_MAX_NEIGH + t];
        sj[t] = j;
        se[t][0] = (c.x[j] - xi) * ih;
        se[t][1] = (c.y[j] - yi) * ih;
        se[t][2] = (c.z[j] - zi) * ih;
    }
    __syncthreads();

    const size_t gs = (size_t)c.gstride;
    double excess = 0.0;
    int flag = 0;
    if (lin < c.nodes)
    {
        const int Nv = c.Nv;
        const double vx = vnode(c.vlo, c.dv, lin % Nv);
        const double vy = vnode(c.vlo, c.dv, (lin / Nv) % Nv);
        const double vz = vnode(c.vlo, c.dv, lin / (Nv * Nv));
        const double *gl = g + lin;
        const double g_self = gl[(size_t)i * gs];
        double out = g_self;
        bool gated = false;
        if (BND)
        {
            double cn = wall_cn3(vx, vy, vz, c.wux[i], c.wuy[i], c.wuz[i], c.wnx[i], c.wny[i],
                                 c.wnz[i]);
            gated = (cn >= 0.0);
        }
        if (!gated)
        {
            // the particle from the foot point, in units of h
            const double ox = (vx - c.mvx[i]) * dt * ih;
            const double oy = (vy - c.mvy[i]) * dt * ih;
            const double oz = (vz - c.mvz[i]) * dt * ih;
            constexpr int NM = P == 10 ? 35 : 10;
            double m[NM], r[P];
#pragma unroll
            for (int q = 0; q < NM; ++q) m[q] = 0.0;
#pragma unroll
            for (int q = 0; q < P; ++q) r[q] = 0.0;
            double gmin = 1e300, gmax = -1e300;
#pragma unroll 2
            for (int t = 0; t < nn; ++t)
            {
                const double gj = gl[(size_t)sj[t] * gs];
                const double x = se[t][0] + ox, y = se[t][1] + oy, z = se[t][2] + oz;
                const double u = fmax(1.0 - (x * x + y * y + z * z), 0.0);
                double w = u * u;                            // mlsWeightSq
                if (w < 1e-30) w = 0.0;
                // a value outside the support must not enter, also if not finite
                mono3_add<P>(w, x, y, z, w > 0.0 ? gj : 0.0, m, r);
                if (DIAG && w > 0.0)
                {
                    gmin = fmin(gmin, gj);
                    gmax = fmax(gmax, gj);
                }
            }
            const double sumW = m[0], sumWG = r[0];
            if (sumW > 0.0)
            {
                double A[P * P];
                fill_matrix<3, P, false>(m, A);
                const bool ok = solve_spd<P>(A, r, tol) && isfinite(r[0]);
                out = ok ? r[0] : sumWG / sumW;
                if (DIAG)
                {
                    if (!ok) flag |= 1;
                    excess = fmax(fmax(out - gmax, gmin - out), 0.0);
                    const bool overshoot = (out < gmin) || (out > gmax);
                    if (overshoot) flag |= 2;
                    if (overshoot && clamp) out = fmin(fmax(out, gmin), gmax);
                }
            }
        }
        gt[(size_t)i * gs + lin] = out;
    }
    if constexpr (DIAG)
    {
        // One flag word and one overshoot sum per workgroup.
        __shared__ double sred[2 * (kBlock / kWave)];
        double red[1] = {excess};
        block_sum<1>(red, sred);
        int f = flag;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) f |= __shfl_xor(f, o, kWave);
        __shared__ int sflag[kBlock / kWave];
        if ((threadIdx.x & (kWave - 1)) == 0) sflag[threadIdx.x / kWave] = f;
        __syncthreads();
        if (threadIdx.x == 0)
        {
            int fa = 0;
            for (int q = 0; q < kBlock / kWave; ++q) fa |= sflag[q];
            if (fa && mlsflag) atomicOr(&mlsflag[i], fa);
            if (red[0] > 0.0 && mlsovr)
            {
                double dv3 = c.dv * c.dv * c.dv;
                atomicAdd(&mlsovr[i], red[0] * dv3);
            }
        }
    }
}

// The interior particles il (P basis functions), then the boundary particles bl
// (linear basis), in one launch. dev: the lists' lengths on the device (the
// stencil classification leaves what it cannot share there), else ni and nb.
// The workgroups stride over the (particle, 256 nodes) items, so the grid needs
// no host count.
template <int P, bool DIAG>
__global__ __launch_bounds__(kBlock) void k_transport3d(DevCloud c, const double *__restrict__ g,
                                                        double *__restrict__ gt, double dt,
                                                        double h, double tol, int clamp,
                                                        int *mlsflag, double *mlsovr,
                                                        const int *__restrict__ il, int ni,
                                                        const int *__restrict__ bl, int nb,
                                                        const int *__restrict__ dev,
                                                        int nchunk, const int *__restrict__ only)
{
    __shared__ double se[AB_MAX_NEIGH][4];
    __shared__ int sj[AB_MAX_NEIGH];
    const int nint = (dev ? dev[0] : ni) * nchunk, nall = nint + (dev ? dev[1] : nb) * nchunk;
    for (int item = xcd_remap(blockIdx.x, gridDim.x); item < nall; item += gridDim.x)
    {
        if (item < nint)
        {
            const int i = il[item / nchunk];
            if (only && !only[i]) continue;      // whole block: one particle
            transport3d_item<P, false, DIAG>(c, g, gt, dt, h, tol, clamp, mlsflag, mlsovr, i,
                                             item % nchunk, se, sj);
        }
        else
        {
            const int e = item - nint;
            transport3d_item<4, true, DIAG>(c, g, gt, dt, h, tol, clamp, mlsflag, mlsovr,
                                            bl[e / nchunk], e % nchunk, se, sj);
        }
    }
}

// Gauss elimination with partial pivoting of the full matrix A, both layers'
// right-hand sides; a column whose pivot is below 1e-30 is skipped and its
// unknown set to 0 (the reference's solve, Solver/CudaBackend.cu:262-300). Row
// swaps select between unrolled rows, so A stays in registers.
template <int P>
__device__ __forceinline__ void solve_pivoted(double (&A)[P * P], double (&r1)[P], double (&r2)[P],
                                              double &o1, double &o2)
{
#pragma unroll
    for (int col = 0; col < P; ++col)
    {
        int piv = col;
        double mx = fabs(A[col * P + col]);
#pragma unroll
        for (int row = col + 1; row < P; ++row)
            if (fabs(A[row * P + col]) > mx) { mx = fabs(A[row * P + col]); piv = row; }
#pragma unroll
        for (int row = col + 1; row < P; ++row)
        {
            const bool take = row == piv;
            auto swap = [take](double &u, double &v) {
                const double t = u;
                u = take ? v : u;
                v = take ? t : v;
            };
#pragma unroll
            for (int q = 0; q < P; ++q) swap(A[col * P + q], A[row * P + q]);
            swap(r1[col], r1[row]);
            swap(r2[col], r2[row]);
        }
        const double d = A[col * P + col];
        if (fabs(d) < 1e-30) continue;
#pragma unroll
        for (int row = col + 1; row < P; ++row)
        {
            const double f = A[row * P + col] / d;
#pragma unroll
            for (int q = col; q < P; ++q) A[row * P + q] -= f * A[col * P + q];
            r1[row] -= f * r1[col];
            r2[row] -= f * r2[col];
        }
    }
    double s1[P], s2[P];
#pragma unroll
    for (int row = P - 1; row >= 0; --row)
    {
        double v1 = r1[row], v2 = r2[row];
#pragma unroll
        for (int q = row + 1; q < P; ++q)
        {
            v1 -= A[row * P + q] * s1[q];
            v2 -= A[row * P + q] * s2[q];
        }
        const double d = A[row * P + row];
        s1[row] = fabs(d) > 1e-30 ? v1 / d : 0.0;
        s2[row] = fabs(d) > 1e-30 ? v2 / d : 0.0;
    }
    o1 = s1[0];
    o2 = s2[0];
}

// One item (particle i, 256 nodes) of kCopyGt + kTransportNode, 2-D Chu layers (Solver/CudaBackend.cu:199-300).
// The reference solves by Gauss elimination with partial pivoting. A is
// symmetric positive definite, so elimination without pivoting is as stable
// and gives the same solution to rounding; where a pivot falls below 1e-9 of
// the largest diagonal entry (a stencil that hardly determines the basis)
// the pivoted elimination runs instead, so what it does with a singular
// matrix stays what it was.
template <int P, bool BND>
__device__ __forceinline__ void transport2d_item(const DevCloud &c, const double *__restrict__ g,
                                                 double *__restrict__ gt, double dt, double h,
                                                 int i, int chunk, double (&se)[AB_MAX_NEIGH][2],
                                                 int (&sj)[AB_MAX_NEIGH])
{
    const int lin = chunk * kBlock + threadIdx.x;
    const int nn = c.nneigh[i];
    if (c.inst) h = c.ih[c.inst[i]];
    const double ih = 1.0 / h;
    const double xi = c.x[i], yi = c.y[i];
    for (int t = threadIdx.x; t < nn; t += kBlock)
    {
        const int j = c.neigh[(size_t)i * AB_MAX_NEIGH + t];
        sj[t] = j;
        se[t][0] = (c.x[j] - xi) * ih;
        se[t][1] = (c.y[j] - yi) * ih;
    }
    __syncthreads();
    if (lin >= c.nodes) return;
    const size_t gs = (size_t)c.gstride;
    const int Nv2 = c.nodes;
    const double vx = vnode(c.vlo, c.dv, lin % c.Nv);
    const double vy = vnode(c.vlo, c.dv, lin / c.Nv);
    const double *gl = g + lin;
    double o1 = gl[(size_t)i * gs], o2 = gl[(size_t)i * gs + Nv2];
    bool gated = false;
    if (BND)
    {
        double cn = wall_cn2(vx, vy, c.wux[i], c.wuy[i], c.wnx[i], c.wny[i]);
        gated = (cn >= 0.0);
    }
    if (!gated)
    {
        const double ox = (vx - c.mvx[i]) * dt * ih, oy = (vy - c.mvy[i]) * dt * ih;
        constexpr int NM = P == 6 ? 15 : 6;
        double m[NM], r1[P], r2[P];
#pragma unroll
        for (int q = 0; q < NM; ++q) m[q] = 0.0;
#pragma unroll
        for (int q = 0; q < P; ++q) { r1[q] = 0.0; r2[q] = 0.0; }
#pragma unroll 2
        for (int t = 0; t < nn; ++t)
        {
            const double *gj = gl + (size_t)sj[t] * gs;
            double g1 = gj[0], g2 = gj[Nv2];
            const double x = se[t][0] + ox, y = se[t][1] + oy;
            const double u = fmax(1.0 - (x * x + y * y), 0.0);
            double w = u * u;                                 // mlsWeight
            // a value outside the support must not enter, also if not finite
            if (w < 1e-30) w = g1 = g2 = 0.0;
            const double wx = w * x, wy = w * y;
            m[0] += w; m[1] += wx; m[2] += wy;
            r1[0] += w * g1; r1[1] += wx * g1; r1[2] += wy * g1;
            r2[0] += w * g2; r2[1] += wx * g2; r2[2] += wy * g2;
            if constexpr (P < 6) { m[3] += wx * x; m[4] += wx * y; m[5] += wy * y; }
            else
            {
                const double xx = wx * x, xy = wx * y, yy = wy * y;
                m[3] += xx; m[4] += xy; m[5] += yy;
                r1[3] += xx * g1; r1[4] += xy * g1; r1[5] += yy * g1;
                r2[3] += xx * g2; r2[4] += xy * g2; r2[5] += yy * g2;
                const double x3 = xx * x, x2y = xx * y, xy2 = xy * y, y3 = yy * y;
                m[6] += x3; m[7] += x2y; m[8] += xy2; m[9] += y3;
                m[10] += x3 * x; m[11] += x3 * y; m[12] += x2y * y; m[13] += xy2 * y;
                m[14] += y3 * y;
            }
        }
        if (m[0] > 0.0)
        {
            double A[P * P];
            fill_matrix<2, P, false>(m, A);
            double dmax = 0.0;
#pragma unroll
            for (int k = 0; k < P; ++k) dmax = fmax(dmax, A[k * P + k]);
            bool ok = true;
            double inv[P], q1[P], q2[P];
#pragma unroll
            for (int k = 0; k < P; ++k) { q1[k] = r1[k]; q2[k] = r2[k]; }
#pragma unroll
            for (int k = 0; k < P; ++k)
            {
                const double d = A[k * P + k];
                ok = ok && (d > 1e-9 * dmax);
                inv[k] = 1.0 / (ok ? d : 1.0);
#pragma unroll
                for (int a = k + 1; a < P; ++a)
                {
                    const double f = A[k * P + a] * inv[k];
#pragma unroll
                    for (int q = a; q < P; ++q) A[a * P + q] -= f * A[k * P + q];
                    q1[a] -= f * q1[k];
                    q2[a] -= f * q2[k];
                }
            }
#pragma unroll
            for (int k = P - 1; k >= 0; --k)
            {
                double v1 = q1[k], v2 = q2[k];
#pragma unroll
                for (int a = k + 1; a < P; ++a)
                {
                    v1 -= A[k * P + a] * q1[a];
                    v2 -= A[k * P + a] * q2[a];
                }
                q1[k] = v1 * inv[k];
                q2[k] = v2 * inv[k];
            }
            o1 = q1[0];
            o2 = q2[0];
            if (!ok)
            {
                double B[P * P];
                fill_matrix<2, P, true>(m, B);
                solve_pivoted<P>(B, r1, r2, o1, o2);
            }
        }
    }
    gt[(size_t)i * gs + lin] = o1;
    gt[(size_t)i * gs + lin + Nv2] = o2;
}

// The interior particles il (P basis functions), then the boundary particles bl
// (linear basis), in one launch: on a small cloud the boundary's own launch
// would cost as much again as its work.
template <int P>
__global__ __launch_bounds__(kBlock) void k_transport2d(DevCloud c, const double *__restrict__ g,
                                                        double *__restrict__ gt, double dt,
                                                        double h, const int *__restrict__ il,
                                                        int ni, const int *__restrict__ bl,
                                                        int nchunk, const int *__restrict__ only)
{
    __shared__ double se[AB_MAX_NEIGH][2];
    __shared__ int sj[AB_MAX_NEIGH];
    const int b = xcd_remap(blockIdx.x, gridDim.x), p = b / nchunk, chunk = b % nchunk;
    if (p < ni)
    {
        const int i = il[p];
        if (only && !only[i]) return;            // whole block: one particle
        transport2d_item<P, false>(c, g, gt, dt, h, i, chunk, se, sj);
    }
    else transport2d_item<3, true>(c, g, gt, dt, h, bl[p - ni], chunk, se, sj);
}

}  // namespace

void launch_transport_fp64(const DevCloud &c, const double *g, double *gt, double dt, double h,
                           int order, double tol, int clamp, int *mlsflag, double *mlsovr,
                           const int *il, int ni, const int *bl, int nb, bool diag, hipStream_t s,
                           const int *only, const int *dev)
{
    if (ni + nb <= 0) return;
    const int nchunk = (c.nodes + kBlock - 1) / kBlock;
    const int all = (ni + nb) * nchunk;
    if (c.dim == 3)
    {
        // with the counts on the device the grid is what fills the chip, not
        // the lists' upper bounds: most of it would find nothing to do
        const int grid = dev ? std::min(all, kFillBlocks) : all;
        auto go = [&](auto kernel) {
            kernel<<<grid, kBlock, 0, s>>>(c, g, gt, dt, h, tol, clamp, mlsflag, mlsovr, il, ni,
                                           bl, nb, dev, nchunk, only);
        };
        if (order >= 2) { if (diag) go(k_transport3d<10, true>); else go(k_transport3d<10, false>); }
        else { if (diag) go(k_transport3d<4, true>); else go(k_transport3d<4, false>); }
    }
    else if (order >= 2)
        k_transport2d<6><<<all, kBlock, 0, s>>>(c, g, gt, dt, h, il, ni, bl, nchunk, only);
    else
        k_transport2d<3><<<all, kBlock, 0, s>>>(c, g, gt, dt, h, il, ni, bl, nchunk, only);
}

}  // namespace ab
