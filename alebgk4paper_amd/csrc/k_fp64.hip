// k_fp64.hip -- the reference formulation of the ALE-BGK step in FP64 on gfx950
// after its transport (k_mls.hip).
//
// Per-particle stages, fixed-order reductions, fusing reference kernels that
// touch only their own particle:
//   commit_collide3 / 2  kPositivity + kNAD3D + kCommit + kScaleG + kWallBC /
//                 kMoments + kCollisionNode (the continuous collision)
//   limit_commit  kPositivity3D + kNAD3D + kCommit  (+ mass partial) and
//   wall_collide  kScaleG + kWallBC + kMoments + kCollisionNode, where the
//                 discrete collision or the MOOD limiter comes between
//   final         kScaleG + kMoments
// and the global sums stay on the device (no host round trip per rescale).
#include "ab_device.hpp"
#include "ab_dm.hpp"
#include "ab_internal.hpp"

namespace ab {

namespace {

// Per-particle mass partial: sum of g*dv^d over the mass-carrying layer
// (kSumMass3D / kSumMass per-thread part, CudaBackend.cu:391-436).
__global__ __launch_bounds__(kBlock) void k_mass_partials(DevCloud c, const double *__restrict__ g,
                                                          double *__restrict__ pmass)
{
    __shared__ double sh[kBlock / kWave];
    const int i = xcd_remap(blockIdx.x, gridDim.x);
    const double dvd = (c.dim == 3) ? c.dv * c.dv * c.dv : c.dv * c.dv;
    const double *p = g + (size_t)i * c.gstride;
    double m[1] = {0.0};
    for (int k = threadIdx.x; k < c.nodes; k += kBlock) m[0] += p[k] * dvd;
    block_sum<1>(m, sh);
    if (threadIdx.x == 0) pmass[i] = m[0];
}

// A particle without mass keeps its moments; its Maxwellian then does not scale
// with the rows, and the end-of-step factor, which holds s1, rescales it by that
// too much: the share it lacks until then.
__device__ __forceinline__ double kept_share(double s1) { return s1 != 0.0 ? 1.0 / s1 - 1.0 : 0.0; }
// The Maxwellian's part of a collided value (or mass) f whose relaxed part is r;
// where f is not finite it stays as it is.
__device__ __forceinline__ double kept_part(double f, double r)
{
    return isfinite(f - r) ? f - r : 0.0;
}
__device__ __forceinline__ bool no_mass(double m) { return !(m > 1e-30); }

// Fixed-order sum of the per-particle partials and the rescale factor
// (sumMassHost + the scalar logic of cudaStep :1627, :1706-1710, :1773-1780),
// kept on the device so no host synchronisation is needed.
// With seg, block k sums instance k's particles seg[k] .. seg[k+1]-1 into
// its scalars (S_COUNT apart) in the same order as a cloud of its own.
__global__ __launch_bounds__(1024) void k_reduce_mass(int N, const double *__restrict__ pmass,
                                                      double *scal, int mode, int nofix,
                                                      const int *__restrict__ seg,
                                                      const double *__restrict__ pnew,
                                                      const double *__restrict__ pold,
                                                      const unsigned char *__restrict__ bnd,
                                                      double coeff)
{
    __shared__ double sh[1024 / kWave], shn[1024 / kWave], sho[1024 / kWave], shk[1024 / kWave];
    int lo = 0, hi = N;
    if (seg)
    {
        lo = seg[blockIdx.x];
        hi = seg[blockIdx.x + 1];
        scal += (size_t)blockIdx.x * S_COUNT;
    }
    double sk = 0.0;               // mass of the Maxwellians that do not scale
    auto add_kept = [&](double v, double m, bool wall) {
        if (no_mass(v) && !wall) sk += kept_part(m, coeff * v);
    };
    // eight loads in flight per thread while eight are left: the one workgroup
    // is bound by their latency (64,000 particles: 29 -> 21 us)
    auto total = [&](const double *__restrict__ p, bool kept) {
        constexpr int U = 8;
        double t = 0.0;
        int i = lo + (int)threadIdx.x;
        for (; i + (U - 1) * 1024 < hi; i += U * 1024)
        {
            double v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = p[i + u * 1024];
#pragma unroll
            for (int u = 0; u < U; ++u) t += v[u];
            if (!kept) continue;
            bool any = false;
#pragma unroll
            for (int u = 0; u < U; ++u) any = any || no_mass(v[u]);
            if (any)
#pragma unroll 1
                for (int k = i; k <= i + (U - 1) * 1024; k += 1024) add_kept(p[k], pmass[k], bnd[k]);
        }
        for (; i < hi; i += 1024)
        {
            // (all three loaded at once: a small cloud's sum is one round trip)
            const double v = p[i], m = kept ? pmass[i] : 0.0;
            const bool wall = kept && bnd[i];
            t += v;
            if (kept) add_kept(v, m, wall);
        }
        return t;
    };
    double s = total(pmass, false), sn = pnew ? total(pnew, bnd != nullptr) : 0.0,
           so = pold ? total(pold, false) : 0.0;
    s = wave_sum(s);
    sn = wave_sum(sn);
    so = wave_sum(so);
    if (__any(sk != 0.0)) sk = wave_sum(sk);
    if ((threadIdx.x & (kWave - 1)) == 0)
    {
        shk[threadIdx.x / kWave] = sk;
        sh[threadIdx.x / kWave] = s;
        shn[threadIdx.x / kWave] = sn;
        sho[threadIdx.x / kWave] = so;
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        double t = 0.0, tn = 0.0, to = 0.0, tk = 0.0;
        for (int q = 0; q < 1024 / kWave; ++q) { t += sh[q]; tn += shn[q]; to += sho[q]; tk += shk[q]; }
        if (mode == R_MASS_FUSED)
        {
            // massOld / massNew, the collided mass after that rescale, and the
            // one end-of-step factor that the unscaled collided rows need:
            // massOld / massColl * massOld / massNew = massOld / t
            const double s1 = (tn > 1e-30) ? to / tn : 1.0;
            if (tk != 0.0) t += tk * kept_share(s1);
            scal[S_MASS_OLD] = to;
            scal[S_MASS_NEW] = tn;
            scal[S_SCALE1] = s1;
            scal[S_MASS_COLL] = s1 * t;
            scal[S_SCALE2] = (!nofix && s1 * t > 1e-30) ? to / t : s1;
        }
        else if (mode == R_MASS_OLD)
            scal[S_MASS_OLD] = t;
        else if (mode == R_MASS_NEW)
        {
            scal[S_MASS_NEW] = t;
            scal[S_SCALE1] = (t > 1e-30) ? scal[S_MASS_OLD] / t : 1.0;
        }
        else
        {
            scal[S_MASS_COLL] = t;
            scal[S_SCALE2] = (!nofix && t > 1e-30) ? scal[S_MASS_OLD] / t : 1.0;
        }
    }
}

// kPositivity3D + kNAD3D + kCommit (CudaBackend.cu:882-954, 328-336) of the
// step with the discrete collision. Writes the committed g, the
// limiter bits and the particle's mass.
__global__ __launch_bounds__(kBlock) void k_limit_commit(DevCloud c, double *__restrict__ g,
                                                         const double *__restrict__ gt,
                                                         const double *__restrict__ rho,
                                                         double *__restrict__ limflag,
                                                         double *__restrict__ pmass)
{
    const int i = xcd_remap(blockIdx.x, gridDim.x) * (kBlock / kWave) + (int)(threadIdx.x / kWave);
    if (i >= c.N) return;                              // whole wave: one particle
    const int lane = threadIdx.x & (kWave - 1);
    const size_t gs = (size_t)c.gstride;
    double *gp = g + (size_t)i * gs;
    const double *tp = gt + (size_t)i * gs;
    const int nodes = c.nodes;
    double flag = 0.0;
    double sc = 1.0, sc2 = 1.0;
    bool fires = false, nad = false;

    const double dv3 = c.dv * c.dv * c.dv;
    double r[3] = {0.0, 0.0, 0.0};             // mPos, mNeg, mFallback
    for (int k = lane; k < nodes; k += kWave)
    {
        double v = tp[k];
        if (v >= 0) r[0] += v;
        else { r[1] += v; r[2] += gp[k]; }
    }
    wave_sums<3>(r);
    fires = (r[1] < -1e-30 && (r[0] + r[1]) > 0);
    if (fires)
    {
        flag += 1.0;
        double target = r[0] + r[1], replaced = r[0] + r[2];
        sc = (replaced > 1e-30) ? target / replaced : 0.0;
    }
    if (!c.bnd[i])
    {
        double rn[1] = {0.0};
        for (int k = lane; k < nodes; k += kWave)
        {
            double v = tp[k];
            if (fires) v = ((v < 0.0) ? gp[k] : v) * sc;
            rn[0] += v;
        }
        wave_sums<1>(rn);
        const double rho_new = rn[0] * dv3;
        const int nn = c.nneigh[i];
        double rmin = 1e300, rmax = -1e300;
        for (int k = lane; k < nn; k += kWave)
        {
            double q = rho[c.neigh[(size_t)i * AB_MAX_NEIGH + k]];
            rmin = fmin(rmin, q);
            rmax = fmax(rmax, q);
        }
        rmin = wave_min(rmin);
        rmax = wave_max(rmax);
        if (!(rmin > rmax))
        {
            double slack = 0.1 * fmax(rmax - rmin, 1e-12) + 1e-9;
            double lo = rmin - slack, hi = rmax + slack;
            if (rho_new > hi && rho_new > 1e-30) { nad = true; sc2 = hi / rho_new; }
            else if (rho_new < lo && rho_new > 1e-30) { nad = true; sc2 = lo / rho_new; }
            if (nad) flag += 2.0;
        }
    }
    double m[1] = {0.0};
    for (int k = lane; k < nodes; k += kWave)
    {
        double v = tp[k];
        if (fires) v = ((v < 0.0) ? gp[k] : v) * sc;
        if (nad) v *= sc2;
        gp[k] = v;
        m[0] += v * dv3;
    }
    wave_sums<1>(m);
    if (lane == 0) { pmass[i] = m[0]; limflag[i] = flag; }
}

// kScaleG (massOld/massNew) + kWallBC3D / kMoments3D + kCollisionNode3D
// (CudaBackend.cu:478-485, 956-1030, 532-569, 1181-1197) and their 2-D
// twins (:338-389, 124-158, 1165-1179). The scale is applied as the value is
// read, which rounds exactly as the stored product would.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_wall_collide(DevCloud c, DmArgs dm, double *__restrict__ g,
                                                         const double *__restrict__ scal,
                                                         double dt, double tau, double R,
                                                         double *rho, double *ux, double *uy,
                                                         double *uz, double *T,
                                                         double *__restrict__ pmass,
                                                         const int *__restrict__ guard)
{
    const int i = xcd_remap(blockIdx.x, gridDim.x) * (kBlock / kWave) + (int)(threadIdx.x / kWave);
    if (i >= c.N) return;                              // whole wave: one particle
    const int lane = threadIdx.x & (kWave - 1);
    if (guard && (!*guard || c.bnd[i])) return;        // whole wave: one particle
    if (c.inst) scal += (size_t)c.inst[i] * S_COUNT;
    const double s1 = scal[S_SCALE1];
    const bool doScale = !guard && scal[S_MASS_NEW] > 1e-30;
    const size_t gs = (size_t)c.gstride;
    double *gp = g + (size_t)i * gs;
    const int nodes = c.nodes, Nv = c.Nv;
    const double dvd = (DIM == 3) ? c.dv * c.dv * c.dv : c.dv * c.dv;
    double m[1] = {0.0};

    if (c.bnd[i])
    {
        const double nx = c.wnx[i], ny = c.wny[i], nz = (DIM == 3) ? c.wnz[i] : 0.0;
        const double Uwx = c.wux[i], Uwy = c.wuy[i], Uwz = (DIM == 3) ? c.wuz[i] : 0.0;
        const double Tw = c.wt[i];
        const double RT2w = 2.0 * R * Tw;
        const double norm = (DIM == 3) ? pow(AB_PI * RT2w, 1.5) : (AB_PI * RT2w);
        double r[2] = {0.0, 0.0};                  // intM, intP
        for (int k = lane; k < nodes; k += kWave)
        {
            double vx = vnode(c.vlo, c.dv, k % Nv);
            double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double vz = (DIM == 3) ? vnode(c.vlo, c.dv, k / (Nv * Nv)) : 0.0;
            double v = doScale ? gp[k] * s1 : gp[k];
            double cn = (DIM == 3) ? wall_cn3(vx, vy, vz, Uwx, Uwy, Uwz, nx, ny, nz)
                                   : wall_cn2(vx, vy, Uwx, Uwy, nx, ny);
            if (cn < 0.0) r[0] += cn * v * dvd;
            else if (cn > 0.0)
            {
                double e2 = (DIM == 3) ? (vx - Uwx) * (vx - Uwx) + (vy - Uwy) * (vy - Uwy)
                                             + (vz - Uwz) * (vz - Uwz)
                                       : (vx - Uwx) * (vx - Uwx) + (vy - Uwy) * (vy - Uwy);
                double Mw = exp(-(e2) / RT2w) / norm;
                r[1] += cn * Mw * dvd;
            }
        }
        wave_sums<2>(r);
        const double rho_w = (r[1] > 1e-30) ? (-r[0] / r[1]) : 1.0;
        for (int k = lane; k < nodes; k += kWave)
        {
            double vx = vnode(c.vlo, c.dv, k % Nv);
            double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double vz = (DIM == 3) ? vnode(c.vlo, c.dv, k / (Nv * Nv)) : 0.0;
            double v = doScale ? gp[k] * s1 : gp[k];
            double v2 = 0.0;
            if constexpr (DIM == 2) v2 = doScale ? gp[k + nodes] * s1 : gp[k + nodes];
            double cn = (DIM == 3) ? wall_cn3(vx, vy, vz, Uwx, Uwy, Uwz, nx, ny, nz)
                                   : wall_cn2(vx, vy, Uwx, Uwy, nx, ny);
            if (cn > 0.0)
            {
                double e2 = (DIM == 3) ? (vx - Uwx) * (vx - Uwx) + (vy - Uwy) * (vy - Uwy)
                                             + (vz - Uwz) * (vz - Uwz)
                                       : (vx - Uwx) * (vx - Uwx) + (vy - Uwy) * (vy - Uwy);
                v = rho_w * exp(-(e2) / RT2w) / norm;
                if constexpr (DIM == 2) v2 = 0.5 * R * Tw * v;
            }
            gp[k] = v;
            if constexpr (DIM == 2) gp[k + nodes] = v2;
            m[0] += v * dvd;
        }
        if (lane == 0)
        {
            rho[i] = rho_w; ux[i] = Uwx; uy[i] = Uwy; T[i] = Tw;
            if (DIM == 3) uz[i] = Uwz;
        }
    }
    else
    {
        double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        for (int k = lane; k < nodes; k += kWave)
        {
            double vx = vnode(c.vlo, c.dv, k % Nv);
            double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double f = doScale ? gp[k] * s1 : gp[k];
            if constexpr (DIM == 3)
            {
                double vz = vnode(c.vlo, c.dv, k / (Nv * Nv));
                r[0] += f * dvd;
                r[1] += vx * f * dvd;
                r[2] += vy * f * dvd;
                r[3] += vz * f * dvd;
                r[4] += (vx * vx + vy * vy + vz * vz) * f * dvd;
            }
            else
            {
                double f2 = doScale ? gp[k + nodes] * s1 : gp[k + nodes];
                r[0] += f * dvd;
                r[1] += vx * f * dvd;
                r[2] += vy * f * dvd;
                r[4] += (vx * vx + vy * vy) * f * dvd + 2.0 * f2 * dvd;
            }
        }
        wave_sums<5>(r);
        double mrho = rho[i], mux = ux[i], muy = uy[i], muz = (DIM == 3) ? uz[i] : 0.0, mT = T[i];
        if (r[0] > 1e-30)
        {
            mrho = r[0];
            mux = r[1] / r[0];
            muy = r[2] / r[0];
            double u2;
            if constexpr (DIM == 3) { muz = r[3] / r[0]; u2 = mux * mux + muy * muy + muz * muz; }
            else u2 = mux * mux + muy * muy;
            double t1 = (r[4] / r[0] - u2) / (3.0 * R);
            mT = t1 > 1e-6 ? t1 : 1e-6;
        }
        const double lam = dt / tau, coeff = 1.0 / (1.0 + lam);
        // discrete-Maxwellian target: Newton on a from the continuous guess
        double a[5] = {0, 0, 0, 0, 0};
        bool useDm = false;
        if constexpr (DIM == 3)
        {
            if (dm.on && r[0] > 1e-30)
            {
                useDm = true;
                const double cs = dm.cs;
                double ac[5];
                dm_guess(mrho, mux, muy, muz, mT, R, cs, ac);
                const float feat[kMlpIn] = {float(mux / cs), float(muy / cs), float(muz / cs),
                                            float(R * mT / (cs * cs)), float(c.dv / cs)};
                float da[kMlpOut] = {0, 0, 0, 0, 0};
                if (dm.mlp) mlp_wave_forward(dm.wb, dm.pf, feat, da);
#pragma unroll
                for (int q = 0; q < 5; ++q) a[q] = ac[q] + (double)da[q];
                const double ms[5] = {r[0], r[1] / cs, r[2] / cs, r[3] / cs, r[4] / (cs * cs)};
                int pass = 0;
                double res = 0.0;
                bool ok = true;
                for (;;)
                {
                    ++pass;
                    double S[15];
#pragma unroll
                    for (int q = 0; q < 15; ++q) S[q] = 0.0;
                    for (int k = lane; k < nodes; k += kWave)
                    {
                        const double xx = vnode(c.vlo, c.dv, k % Nv) / cs;
                        const double yy = vnode(c.vlo, c.dv, (k / Nv) % Nv) / cs;
                        const double zz = vnode(c.vlo, c.dv, k / (Nv * Nv)) / cs;
                        const double e = exp(a[0] + a[1] * xx + a[2] * yy + a[3] * zz
                                             + a[4] * (xx * xx + yy * yy + zz * zz)) * dvd;
                        dm_accum(S, e, xx, yy, zz);
                    }
                    wave_sums<15>(S);
                    double F[5];
                    res = 0.0;
#pragma unroll
                    for (int q = 0; q < 5; ++q) { F[q] = S[q] - ms[q]; res = fmax(res, fabs(F[q])); }
                    res /= fabs(ms[0]);
                    if (res <= dm.tol || pass > dm.maxit) break;
                    double d[5];
                    if (!dm_solve5(S, F, d)) { ok = false; break; }
#pragma unroll
                    for (int q = 0; q < 5; ++q) a[q] -= d[q];
                }
                bool conv = ok && res <= dm.tol;
#pragma unroll
                for (int q = 0; q < 5; ++q) conv = conv && isfinite(a[q]);
                if (!conv)
#pragma unroll
                    for (int q = 0; q < 5; ++q) a[q] = ac[q];       // continuous fallback
                if (lane == 0)
                {
#pragma unroll
                    for (int q = 0; q < 5; ++q) dm.alpha[(size_t)i * 5 + q] = a[q];
                    dm.passes[i] = conv ? pass : dm.maxit + 2;
                    dm.res[i] = res;
                    if (dm.rec)
                    {
                        float *row = dm.rec + (size_t)i * kMlpRow;
#pragma unroll
                        for (int q = 0; q < kMlpIn; ++q) row[q] = feat[q];
#pragma unroll
                        for (int q = 0; q < kMlpOut; ++q) row[kMlpIn + q] = float(a[q] - ac[q]);
                        row[kMlpIn + kMlpOut] = conv ? 1.0f : 0.0f;
                    }
                }
            }
        }
        for (int k = lane; k < nodes; k += kWave)
        {
            double vx = vnode(c.vlo, c.dv, k % Nv);
            double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double f = doScale ? gp[k] * s1 : gp[k];
            if constexpr (DIM == 3)
            {
                double vz = vnode(c.vlo, c.dv, k / (Nv * Nv));
                double M;
                if (useDm)
                {
                    const double xx = vx / dm.cs, yy = vy / dm.cs, zz = vz / dm.cs;
                    M = exp(a[0] + a[1] * xx + a[2] * yy + a[3] * zz
                            + a[4] * (xx * xx + yy * yy + zz * zz));
                }
                else M = maxwellian3d(vx, vy, vz, mux, muy, muz, mT, mrho, R);
                f = coeff * (f + lam * M);
            }
            else
            {
                double f2 = doScale ? gp[k + nodes] * s1 : gp[k + nodes];
                double Mg1 = maxwellian_g1(vx, vy, mux, muy, mT, mrho, R);
                f = coeff * (f + lam * Mg1);
                f2 = coeff * (f2 + lam * 0.5 * R * mT * Mg1);
                gp[k + nodes] = f2;
            }
            gp[k] = f;
            m[0] += f * dvd;
        }
        if (lane == 0)
        {
            rho[i] = mrho; ux[i] = mux; uy[i] = muy; T[i] = mT;
            if (DIM == 3) uz[i] = muz;
        }
    }
    wave_sums<1>(m);
    if (lane == 0) pmass[i] = m[0];
}

// kPositivity + kCommit + kScaleG + kWallBC / kMoments + kCollisionNode of
// the 2-D step (CudaBackend.cu:304-336, 478-485, 338-389, 124-158,
// 1165-1179) in one pass per particle for the 2-D table formulation: gt is
// read (the row stays in cache between the passes over it) and the collided
// g written once, where k_limit_commit<2> and k_wall_collide<2> read and
// write g twice. The rescale between commit and collision is left out: the
// wall density, the density moment and the Maxwellians scale with g, u and
// T do not, so the collided row of the unscaled commit is the collided row
// of the rescaled one divided by massOld / massNew. The reduction then takes
// the committed masses (pnew) and the collided masses (pmass) and gives
// k_final the one factor that the rows need; the wall densities get the
// first factor there. A particle without mass keeps its moments and a wall that
// emits nothing has density 1, whatever the rescale: the reduction and k_final
// make up for it (FusedFinal). Results agree with the separate kernels to rounding.
// U > 0: rows of at most U * 64 nodes (Nv <= 16 for U = 4), which each lane
// loads into registers once (U values of each layer); U == 0: any row, read
// again from memory in every pass. Both sum in the same order, so they give
// identical results.
template <int U>
__global__ __launch_bounds__(kBlock) void k_commit_collide2(DevCloud c, double *__restrict__ g,
                                                            double *__restrict__ gt,
                                                            double dt, double tau, double R,
                                                            double *rho, double *ux, double *uy,
                                                            double *T, double *__restrict__ limflag,
                                                            double *__restrict__ pnew,
                                                            double *__restrict__ pmass)
{
    const int i = xcd_remap(blockIdx.x, gridDim.x) * (kBlock / kWave) + (int)(threadIdx.x / kWave);
    if (i >= c.N) return;                              // whole wave: one particle
    const int lane = threadIdx.x & (kWave - 1);
    const size_t gs = (size_t)c.gstride;
    double *gp = g + (size_t)i * gs, *tp = gt + (size_t)i * gs;
    const int nodes = c.nodes, Nv = c.Nv;
    const double dvd = c.dv * c.dv;
    const int nu = U > 0 ? U : (nodes + kWave - 1) / kWave;   // passes of a wave over the row

    double t1[U > 0 ? U : 1], t2[U > 0 ? U : 1];
    if constexpr (U > 0)
    {
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int k = lane + u * kWave;
            t1[u] = k < nodes ? tp[k] : 0.0;
            t2[u] = k < nodes ? tp[k + nodes] : 0.0;
        }
    }
    auto raw1 = [&](int u, int k) { if constexpr (U > 0) return t1[u]; else return tp[k]; };
    auto raw2 = [&](int u, int k) { if constexpr (U > 0) return t2[u]; else return tp[k + nodes]; };

    double rp[2] = {0.0, 0.0};                     // mPos, mNeg of g1
#pragma unroll
    for (int u = 0; u < nu; ++u)
    {
        const int k = lane + u * kWave;
        if (k >= nodes) continue;
        const double v = raw1(u, k);
        if (v >= 0) rp[0] += v; else rp[1] += v;
    }
    wave_sums<2>(rp);
    const bool fires = (rp[1] < -1e-30 && rp[0] > 1e-30 && (rp[0] + rp[1]) > 0);
    const double sc = fires ? (rp[0] + rp[1]) / rp[0] : 1.0;
    auto committed = [&](int u, int k, double &v1, double &v2) {
        v1 = raw1(u, k);
        v2 = raw2(u, k);
        if (fires)
        {
            if (v1 < 0) { v1 = 0; v2 = 0; }
            else { v1 *= sc; v2 *= sc; }
        }
    };
    double m[1] = {0.0};
    double mnew = 0.0, flag = fires ? 1.0 : 0.0;

    if (c.bnd[i])
    {
        const double nx = c.wnx[i], ny = c.wny[i];
        const double Uwx = c.wux[i], Uwy = c.wuy[i];
        const double Tw = c.wt[i];
        const double RT2w = 2.0 * R * Tw;
        const double norm = AB_PI * RT2w;
        double r[3] = {0.0, 0.0, 0.0};             // intM, intP, committed mass
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            const double vx = vnode(c.vlo, c.dv, k % Nv);
            const double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double v, v2;
            committed(u, k, v, v2);
            const double cn = wall_cn2(vx, vy, Uwx, Uwy, nx, ny);
            if (cn < 0.0) r[0] += cn * v * dvd;
            else if (cn > 0.0)
            {
                const double e2 = (vx - Uwx) * (vx - Uwx) + (vy - Uwy) * (vy - Uwy);
                const double Mw = exp(-(e2) / RT2w) / norm;
                r[1] += cn * Mw * dvd;
            }
            r[2] += v * dvd;
        }
        wave_sums<3>(r);
        const double rho_w = (r[1] > 1e-30) ? (-r[0] / r[1]) : 1.0;
        if (!(r[1] > 1e-30)) flag += kNoEmission;
        mnew = r[2];
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            const double vx = vnode(c.vlo, c.dv, k % Nv);
            const double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double v, v2;
            committed(u, k, v, v2);
            const double cn = wall_cn2(vx, vy, Uwx, Uwy, nx, ny);
            if (cn > 0.0)
            {
                const double e2 = (vx - Uwx) * (vx - Uwx) + (vy - Uwy) * (vy - Uwy);
                v = rho_w * exp(-(e2) / RT2w) / norm;
                v2 = 0.5 * R * Tw * v;
            }
            gp[k] = v;
            gp[k + nodes] = v2;
            m[0] += v * dvd;
        }
        if (lane == 0) { rho[i] = rho_w; ux[i] = Uwx; uy[i] = Uwy; T[i] = Tw; }
    }
    else
    {
        double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            const double vx = vnode(c.vlo, c.dv, k % Nv);
            const double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double f, f2;
            committed(u, k, f, f2);
            r[0] += f * dvd;
            r[1] += vx * f * dvd;
            r[2] += vy * f * dvd;
            r[4] += (vx * vx + vy * vy) * f * dvd + 2.0 * f2 * dvd;
        }
        wave_sums<5>(r);
        mnew = r[0];
        double mrho = rho[i], mux = ux[i], muy = uy[i], mT = T[i];
        const bool kept = no_mass(r[0]);
        if (!kept)
        {
            mrho = r[0];
            mux = r[1] / r[0];
            muy = r[2] / r[0];
            const double t1m = (r[4] / r[0] - (mux * mux + muy * muy)) / (3.0 * R);
            mT = t1m > 1e-6 ? t1m : 1e-6;
        }
        const double lam = dt / tau, coeff = 1.0 / (1.0 + lam);
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            const double vx = vnode(c.vlo, c.dv, k % Nv);
            const double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            double f, f2;
            committed(u, k, f, f2);
            if (kept && fires) { tp[k] = f; tp[k + nodes] = f2; }      // for k_final
            const double Mg1 = maxwellian_g1(vx, vy, mux, muy, mT, mrho, R);
            f = coeff * (f + lam * Mg1);
            f2 = coeff * (f2 + lam * 0.5 * R * mT * Mg1);
            gp[k] = f;
            gp[k + nodes] = f2;
            m[0] += f * dvd;
        }
        if (lane == 0) { rho[i] = mrho; ux[i] = mux; uy[i] = muy; T[i] = mT; }
    }
    wave_sums<1>(m);
    if (lane == 0)
    {
        pmass[i] = m[0];
        pnew[i] = mnew;
        limflag[i] = flag;
    }
}

// The 3-D step's kPositivity3D + kNAD3D + kCommit + kScaleG + kWallBC3D /
// kMoments3D + kCollisionNode3D (CudaBackend.cu:882-954, 328-336, 478-485,
// 956-1030, 532-569, 1181-1197) in one pass per particle, one wave each, with
// the rescale between commit and collision left to the end of the step as in
// k_commit_collide2 (wall density, moments and Maxwellians scale with g). The
// row is read once and the collided one written once; k_limit_commit<3> and
// k_wall_collide<3> read three rows and wrote two. What bounded those beside
// the traffic was an FP64 exponential per node: the velocity grid is a tensor
// product, so exp(-|v - u|^2 / 2RT) is the product of three factors, 3 Nv
// exponentials a particle. 40^3 / Nv 10: 332 + 686 -> 286 us, 3.6 TB/s of its one
// read and one write.
//
// NAD compares with the neighbours' densities of the step's start, which must
// not change while other particles still read them: the wall densities go to
// rho_wall, and k_final writes rho.
// U > 0: rows of at most U * 64 nodes stay in registers; U == 0: any row, read
// again from the cache in each pass, in the same order of sums.
// mg1, mg2: ceil(2^32 / Nv), ceil(2^32 / Nv^2), exact quotients for k < Nv^3.
template <int U>
__global__ __launch_bounds__(kBlock) void k_commit_collide3(
    DevCloud c, double *__restrict__ g, double *__restrict__ gt, unsigned mg1, unsigned mg2,
    double dt, double tau, double R, const double *__restrict__ rho, double *__restrict__ rho_wall,
    double *ux, double *uy, double *uz, double *T, double *__restrict__ limflag,
    double *__restrict__ pnew, double *__restrict__ pmass)
{
    __shared__ double tab[kBlock / kWave][3][kMaxNv];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int i = xcd_remap(blockIdx.x, gridDim.x) * (kBlock / kWave) + w;
    if (i >= c.N) return;                              // whole wave: one particle
    const size_t gs = (size_t)c.gstride;
    double *gp = g + (size_t)i * gs, *tp = gt + (size_t)i * gs;
    const int nodes = c.nodes, Nv = c.Nv;
    const double dv3 = c.dv * c.dv * c.dv;
    const int nu = U > 0 ? U : (nodes + kWave - 1) / kWave;

    double t[U > 0 ? U : 1];
    if constexpr (U > 0)
    {
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int k = lane + u * kWave;
            t[u] = k < nodes ? tp[k] : 0.0;
        }
    }
    const bool wall = c.bnd[i];
    // the neighbours' densities while the row is on its way
    double rmin = 1e300, rmax = -1e300;
    if (!wall)
    {
        const int nn = c.nneigh[i];
        for (int k = lane; k < nn; k += kWave)
        {
            const double q = rho[c.neigh[(size_t)i * AB_MAX_NEIGH + k]];
            rmin = fmin(rmin, q);
            rmax = fmax(rmax, q);
        }
    }
    double r[3] = {0.0, 0.0, 0.0};                     // mPos, mNeg, mFallback
#pragma unroll
    for (int u = 0; u < nu; ++u)
    {
        const int k = lane + u * kWave;
        if (k >= nodes) continue;
        double v;
        if constexpr (U > 0) v = t[u]; else v = tp[k];
        if (v >= 0) r[0] += v;
        else { r[1] += v; r[2] += gp[k]; }
    }
    wave_sums<3>(r);
    double flag = 0.0, sc = 1.0, sc2 = 1.0;
    const bool fires = (r[1] < -1e-30 && (r[0] + r[1]) > 0);
    if (fires)
    {
        flag += 1.0;
        const double target = r[0] + r[1], replaced = r[0] + r[2];
        sc = (replaced > 1e-30) ? target / replaced : 0.0;
    }
    // the committed value of node k (register u)
    auto committed = [&](int u, int k) {
        double v;
        if constexpr (U > 0) v = t[u]; else v = tp[k];
        if (fires) v = ((v < 0.0) ? gp[k] : v) * sc;
        return v * sc2;
    };
    if (!wall)
    {
        double rn = r[0] + r[1];
        if (fires)
        {
            rn = 0.0;
#pragma unroll
            for (int u = 0; u < nu; ++u)
            {
                const int k = lane + u * kWave;
                if (k < nodes) rn += committed(u, k);
            }
            rn = wave_sum(rn);
        }
        const double rho_new = rn * dv3;
        rmin = wave_min(rmin);
        rmax = wave_max(rmax);
        if (!(rmin > rmax))
        {
            const double slack = 0.1 * fmax(rmax - rmin, 1e-12) + 1e-9;
            const double lo = rmin - slack, hi = rmax + slack;
            bool nad = false;
            if (rho_new > hi && rho_new > 1e-30) { nad = true; sc2 = hi / rho_new; }
            else if (rho_new < lo && rho_new > 1e-30) { nad = true; sc2 = lo / rho_new; }
            if (nad) flag += 2.0;
        }
    }
    if constexpr (U > 0)
    {
        // commit: the later passes read the register
        if (fires || sc2 != 1.0)
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int k = lane + u * kWave;
                if (k < nodes) t[u] = committed(u, k);
            }
    }
    auto value = [&](int u, int k) { if constexpr (U > 0) return t[u]; else return committed(u, k); };
    auto node = [&](int k, int &iv, int &jv, int &kv) {
        kv = (int)__umulhi((unsigned)k, mg2);
        const int p = k - kv * (Nv * Nv);
        jv = (int)__umulhi((unsigned)p, mg1);
        iv = p - jv * Nv;
    };
    // the three factors of exp(-|v - u|^2 / (2RT)), one entry per lane and pass
    auto factors = [&](double ax, double ay, double az, double twoRT) {
        for (int e = lane; e < 3 * Nv; e += kWave)
        {
            const int axis = e / Nv, l = e - axis * Nv;
            const double d = vnode(c.vlo, c.dv, l) - (axis == 0 ? ax : axis == 1 ? ay : az);
            tab[w][axis][l] = exp(-(d * d) / twoRT);
        }
        wave_lds_sync();
    };
    double m = 0.0, mnew = 0.0;
    if (wall)
    {
        const double nx = c.wnx[i], ny = c.wny[i], nz = c.wnz[i];
        const double Ux = c.wux[i], Uy = c.wuy[i], Uz = c.wuz[i], Tw = c.wt[i];
        const double RT2w = 2.0 * R * Tw, in = 1.0 / pow(AB_PI * RT2w, 1.5);
        factors(Ux, Uy, Uz, RT2w);
        double q[3] = {0.0, 0.0, 0.0};                 // intM, intP, committed mass
        auto cn_of = [&](int iv, int jv, int kv) {
            return wall_cn3(vnode(c.vlo, c.dv, iv), vnode(c.vlo, c.dv, jv), vnode(c.vlo, c.dv, kv),
                            Ux, Uy, Uz, nx, ny, nz);
        };
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            int iv, jv, kv;
            node(k, iv, jv, kv);
            const double v = value(u, k), cn = cn_of(iv, jv, kv);
            if (cn < 0.0) q[0] += cn * v;
            else if (cn > 0.0) q[1] += cn * (tab[w][0][iv] * tab[w][1][jv] * tab[w][2][kv]);
            q[2] += v;
        }
        wave_sums<3>(q);
        const double intM = q[0] * dv3, intP = q[1] * in * dv3;
        const double rho_w = (intP > 1e-30) ? (-intM / intP) : 1.0, am = rho_w * in;
        if (!(intP > 1e-30)) flag += kNoEmission;
        mnew = q[2] * dv3;
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            int iv, jv, kv;
            node(k, iv, jv, kv);
            double v = value(u, k);
            if (cn_of(iv, jv, kv) > 0.0) v = am * (tab[w][0][iv] * tab[w][1][jv] * tab[w][2][kv]);
            gp[k] = v;
            m += v;
        }
        if (lane == 0) { rho_wall[i] = rho_w; ux[i] = Ux; uy[i] = Uy; uz[i] = Uz; T[i] = Tw; }
    }
    else
    {
        double q[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            int iv, jv, kv;
            node(k, iv, jv, kv);
            const double vx = vnode(c.vlo, c.dv, iv), vy = vnode(c.vlo, c.dv, jv),
                         vz = vnode(c.vlo, c.dv, kv);
            const double f = value(u, k);
            q[0] += f;
            q[1] += vx * f;
            q[2] += vy * f;
            q[3] += vz * f;
            q[4] += (vx * vx + vy * vy + vz * vz) * f;
        }
        wave_sums<5>(q);
#pragma unroll
        for (int a = 0; a < 5; ++a) q[a] *= dv3;
        mnew = q[0];
        double mrho = rho[i], mux = ux[i], muy = uy[i], muz = uz[i], mT = T[i];
        const bool kept = no_mass(q[0]), repaired = kept && (fires || sc2 != 1.0);
        if (!kept)
        {
            mrho = q[0];
            mux = q[1] / q[0];
            muy = q[2] / q[0];
            muz = q[3] / q[0];
            const double t1 = (q[4] / q[0] - (mux * mux + muy * muy + muz * muz)) / (3.0 * R);
            mT = t1 > 1e-6 ? t1 : 1e-6;
        }
        const double lam = dt / tau, coeff = 1.0 / (1.0 + lam);
        const double twoRT = 2.0 * R * mT, am = lam * mrho / pow(AB_PI * twoRT, 1.5);
        factors(mux, muy, muz, twoRT);
#pragma unroll
        for (int u = 0; u < nu; ++u)
        {
            const int k = lane + u * kWave;
            if (k >= nodes) continue;
            int iv, jv, kv;
            node(k, iv, jv, kv);
            const double v = value(u, k);
            if (repaired) tp[k] = v;                                   // for k_final
            const double f = coeff * (v + am * (tab[w][0][iv] * tab[w][1][jv] * tab[w][2][kv]));
            gp[k] = f;
            m += f;
        }
        if (lane == 0) { ux[i] = mux; uy[i] = muy; uz[i] = muz; T[i] = mT; }
    }
    m = wave_sum(m) * dv3;
    if (lane == 0)
    {
        pmass[i] = m;
        pnew[i] = mnew;
        limflag[i] = flag;
    }
}

// kScaleG (massOld/massColl) + kMoments3D / kMoments (CudaBackend.cu:1773-1788).
// One wave per particle, four per workgroup: each lane loads four nodes of
// both layers before it adds any, and the sums are wave reductions, so a
// row's loads are in flight together and no workgroup barrier is needed.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_final(DevCloud c, double *__restrict__ g,
                                                  const double *__restrict__ scal, double R,
                                                  double *rho, double *ux, double *uy,
                                                  double *uz, double *T,
                                                  double *__restrict__ pmass,
                                                  const int *__restrict__ guard, FusedFinal fu)
{
    constexpr int kPer = kBlock / kWave;
    const int i = xcd_remap(blockIdx.x, gridDim.x) * kPer + (int)(threadIdx.x / kWave);
    if (i >= c.N) return;                          // whole wave
    if (guard && !*guard) return;
    const int lane = threadIdx.x & (kWave - 1);
    if (c.inst) scal += (size_t)c.inst[i] * S_COUNT;
    const double s2 = scal[S_SCALE2];
    const double s1 = scal[S_SCALE1];
    const bool doScale = (s2 != 1.0);
    const size_t gs = (size_t)c.gstride;
    double *gp = g + (size_t)i * gs;
    const int nodes = c.nodes, Nv = c.Nv;
    const double dvd = (DIM == 3) ? c.dv * c.dv * c.dv : c.dv * c.dv;
    const bool inner = !c.bnd[i];
    // (loaded beside the row, looked at once that is there)
    const double mnew = fu.pnew ? fu.pnew[i] : 1.0;
    double r[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};   // rho, rux, ruy, ruz, E, mass
    auto sums = [&](int k, double f, double f2) {
        r[5] += f * dvd;
        if (inner)
        {
            double vx = vnode(c.vlo, c.dv, k % Nv);
            double vy = vnode(c.vlo, c.dv, (k / Nv) % Nv);
            r[0] += f * dvd;
            r[1] += vx * f * dvd;
            r[2] += vy * f * dvd;
            if constexpr (DIM == 3)
            {
                double vz = vnode(c.vlo, c.dv, k / (Nv * Nv));
                r[3] += vz * f * dvd;
                r[4] += (vx * vx + vy * vy + vz * vz) * f * dvd;
            }
            else
                r[4] += (vx * vx + vy * vy) * f * dvd + 2.0 * f2 * dvd;
        }
    };
    auto node = [&](int k, double f, double f2) {
        if (doScale)
        {
            f *= s2; gp[k] = f;
            if constexpr (DIM == 2) { f2 *= s2; gp[k + nodes] = f2; }
        }
        sums(k, f, f2);
    };
    constexpr int U = 4;
    int k0 = 0;
    for (; k0 + U * kWave <= nodes; k0 += U * kWave)
    {
        double f[U], f2[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            f[u] = gp[k0 + u * kWave + lane];
            f2[u] = (DIM == 2) ? gp[k0 + u * kWave + lane + nodes] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) node(k0 + u * kWave + lane, f[u], f2[u]);
    }
    for (int k = k0 + lane; k < nodes; k += kWave)
        node(k, gp[k], (DIM == 2) ? gp[k + nodes] : 0.0);
    if (__any(inner && no_mass(mnew)))                 // whole wave: one particle
    {
        // a particle without mass: the share that its Maxwellian lacks, and the
        // sums again (after the loop: in it the test would wait before the row's
        // loads, or its registers cost a wave)
        const double *tp = fu.gt + (size_t)i * gs;
        const double b = kept_share(s1), sc = s2 * fu.coeff;
#pragma unroll
        for (int q = 0; q < 6; ++q) r[q] = 0.0;
#pragma unroll 1
        for (int k = lane; k < nodes; k += kWave)
        {
            double f = gp[k], f2 = 0.0;
            gp[k] = f += b * kept_part(f, sc * tp[k]);
            if constexpr (DIM == 2)
            {
                f2 = gp[k + nodes];
                gp[k + nodes] = f2 += b * kept_part(f2, sc * tp[k + nodes]);
            }
            sums(k, f, f2);
        }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) r[q] = wave_sum(r[q]);
    if (lane == 0)
    {
        pmass[i] = r[5];
        if (!inner && fu.rho_wall)
        {
            const double lim = fu.limflag[i];
            const bool none = lim >= kNoEmission;
            rho[i] = none ? 1.0 : fu.rho_wall[i] * s1;
            if (none) fu.limflag[i] = lim - kNoEmission;
        }
        if (inner && r[0] > 1e-30)
        {
            double mux = r[1] / r[0], muy = r[2] / r[0], muz = 0.0, u2;
            if constexpr (DIM == 3) { muz = r[3] / r[0]; u2 = mux * mux + muy * muy + muz * muz; }
            else u2 = mux * mux + muy * muy;
            double t1 = (r[4] / r[0] - u2) / (3.0 * R);
            rho[i] = r[0]; ux[i] = mux; uy[i] = muy; T[i] = t1 > 1e-6 ? t1 : 1e-6;
            if (DIM == 3) uz[i] = muz;
        }
        // no mass at the step's end (or none that is a number), and some before
        // the collision: the density is the collision's
        else if (inner && fu.pnew && !no_mass(mnew)) rho[i] = mnew * s1;
    }
}

// ---- the reference's CPU-step limiter (MOOD) ---------------------------------

// The positivity repair inside the CPU transport (MLSTransport/MLSTransport.cpp
// :189-200 in 3-D, :287-307 in 2-D) on one particle's row: negatives to
// zero, the rest scaled to keep the mass (2-D: on g1, g2 following). Returns
// whether it fired (every thread).
template <int DIM>
__device__ __forceinline__ bool positivity_zero(const DevCloud &c, double *p, double *sh)
{
    const int n = c.nodes;
    double r[2] = {0.0, 0.0};                  // mPos, mNeg
    for (int k = threadIdx.x; k < n; k += kBlock)
    {
        const double v = p[k];
        if (v >= 0.0) r[0] += v; else r[1] += v;
    }
    block_sum<2>(r, sh);
    if (!(r[1] < -1e-30 && r[0] > 1e-30 && (r[0] + r[1]) > 0.0)) return false;
    const double sc = (r[0] + r[1]) / r[0];
    for (int k = threadIdx.x; k < n; k += kBlock)
    {
        const bool neg = p[k] < 0.0;
        p[k] = neg ? 0.0 : p[k] * sc;
        if constexpr (DIM == 2) p[k + n] = neg ? 0.0 : p[k + n] * sc;
    }
    __syncthreads();
    return true;
}

// Positivity on every particle's transported row, then checkTransportPAD
// (MLSTransport/MLSTransport.cpp:324-379) on the interior ones: flagged when
// the row's mass is not finite or not positive, or its density leaves the
// neighbours' current range widened by 0.1 of the range (at least 1e-12) plus
// 1e-9. mood[i] = flagged; limflag: +1 positivity, +2 flagged.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_mood_check(DevCloud c, double *__restrict__ gt,
                                                       const double *__restrict__ rho,
                                                       int *__restrict__ mood,
                                                       double *__restrict__ limflag)
{
    __shared__ double sh[2 * (kBlock / kWave)];
    const int i = xcd_remap(blockIdx.x, gridDim.x);
    double *p = gt + (size_t)i * c.gstride;
    const bool fired = positivity_zero<DIM>(c, p, sh);
    bool flag = false;
    if (!c.bnd[i])
    {
        double m[1] = {0.0};
        for (int k = threadIdx.x; k < c.nodes; k += kBlock) m[0] += p[k];
        block_sum<1>(m, sh);
        const double dvN = (DIM == 3) ? c.dv * c.dv * c.dv : c.dv * c.dv;
        flag = !isfinite(m[0]) || m[0] <= 0.0;     // a non-finite value makes the sum non-finite
        const int nn = c.nneigh[i];
        double lo = 1e300, hi = -1e300;
        for (int k = threadIdx.x; k < nn; k += kBlock)
        {
            const double q = rho[c.neigh[(size_t)i * AB_MAX_NEIGH + k]];
            lo = fmin(lo, q); hi = fmax(hi, q);
        }
        block_minmax(lo, hi, sh);
        if (!flag && nn > 0)
        {
            const double rn = m[0] * dvN;
            const double slack = 0.1 * fmax(hi - lo, 1e-12) + 1e-9;
            flag = (rn < lo - slack || rn > hi + slack);
        }
    }
    if (threadIdx.x == 0)
    {
        mood[i] = flag ? 1 : 0;
        limflag[i] = (fired ? 1.0 : 0.0) + (flag ? 2.0 : 0.0);
    }
}

// The flagged particles' rows came from the linear re-transport: positivity
// once more on those (the repair runs inside every transport pass); then the
// commit gt -> g for every particle and its mass partial.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_mood_commit(DevCloud c, double *__restrict__ g,
                                                        double *__restrict__ gt,
                                                        const int *__restrict__ mood,
                                                        double *__restrict__ limflag,
                                                        double *__restrict__ pmass)
{
    __shared__ double sh[2 * (kBlock / kWave)];
    const int i = xcd_remap(blockIdx.x, gridDim.x);
    const size_t gs = (size_t)c.gstride;
    double *tp = gt + (size_t)i * gs;
    double *gp = g + (size_t)i * gs;
    if (mood[i])
    {
        const bool fired = positivity_zero<DIM>(c, tp, sh);
        if (fired && threadIdx.x == 0 && !((int)limflag[i] & 1)) limflag[i] += 1.0;
    }
    const double dvd = (DIM == 3) ? c.dv * c.dv * c.dv : c.dv * c.dv;
    double m[1] = {0.0};
    for (int k = threadIdx.x; k < (int)gs; k += kBlock)
    {
        const double v = tp[k];
        gp[k] = v;
        if (k < c.nodes) m[0] += v * dvd;
    }
    block_sum<1>(m, sh);
    if (threadIdx.x == 0) pmass[i] = m[0];
}

// moodCheck (MomentCalculations/Conservation.cpp:16-38) with padCheck
// (MLSTransport/MLSBasis.hpp:208-222) on the interior particles after the
// collision: rho < 1e-10, T < 1e-6 or a mass-carrying value below -1e-14.
// limflag +4 and *fail set for a failing particle.
__global__ __launch_bounds__(kBlock) void k_pad_check(DevCloud c, const double *__restrict__ g,
                                                      const double *__restrict__ rho,
                                                      const double *__restrict__ T,
                                                      double *__restrict__ limflag,
                                                      int *__restrict__ fail)
{
    __shared__ int sbad[kBlock / kWave];
    const int i = xcd_remap(blockIdx.x, gridDim.x);
    if (c.bnd[i]) return;
    const double *p = g + (size_t)i * c.gstride;
    int bad = 0;
    for (int k = threadIdx.x; k < c.nodes; k += kBlock) bad |= (p[k] < -1.0e-14) ? 1 : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) bad |= __shfl_xor(bad, o, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) sbad[threadIdx.x / kWave] = bad;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        int b = (rho[i] < 1.0e-10 || T[i] < 1.0e-6) ? 1 : 0;
        for (int q = 0; q < kBlock / kWave; ++q) b |= sbad[q];
        if (b)
        {
            limflag[i] += 4.0;
            atomicOr(fail, 1);
        }
    }
}

}  // namespace

void launch_mass_partials(const DevCloud &c, const double *g, double *pmass, hipStream_t s)
{
    k_mass_partials<<<c.N, kBlock, 0, s>>>(c, g, pmass);
}

void launch_reduce_mass(int N, const double *pmass, double *scal, int mode, int nofix,
                        hipStream_t s, const int *seg, int nseg, const double *pnew,
                        const double *pold, const unsigned char *bnd, double coeff)
{
    k_reduce_mass<<<seg ? nseg : 1, 1024, 0, s>>>(N, pmass, scal, mode, nofix, seg, pnew, pold, bnd,
                                                  coeff);
}

void launch_limit_commit(const DevCloud &c, double *g, const double *gt, const double *rho,
                         double *limflag, double *pmass, hipStream_t s)
{
    const int nb = (c.N + kBlock / kWave - 1) / (kBlock / kWave);
    k_limit_commit<<<nb, kBlock, 0, s>>>(c, g, gt, rho, limflag, pmass);
}

void launch_wall_collide(const DevCloud &c, const DmArgs &dm, double *g, const double *scal,
                         double dt, double tau, double R, double *rho, double *ux, double *uy,
                         double *uz, double *T, double *pmass, hipStream_t s, const int *guard)
{
    const int nb = (c.N + kBlock / kWave - 1) / (kBlock / kWave);
    if (c.dim == 3)
        k_wall_collide<3><<<nb, kBlock, 0, s>>>(c, dm, g, scal, dt, tau, R, rho, ux, uy, uz, T,
                                                pmass, guard);
    else
        k_wall_collide<2><<<nb, kBlock, 0, s>>>(c, dm, g, scal, dt, tau, R, rho, ux, uy, uz, T,
                                                pmass, guard);
}

void launch_final(const DevCloud &c, double *g, const double *scal, double R, double *rho,
                  double *ux, double *uy, double *uz, double *T, double *pmass, hipStream_t s,
                  const int *guard, const FusedFinal &fused)
{
    const int nb = (c.N + kBlock / kWave - 1) / (kBlock / kWave);
    if (c.dim == 3)
        k_final<3><<<nb, kBlock, 0, s>>>(c, g, scal, R, rho, ux, uy, uz, T, pmass, guard,
                                         fused);
    else
        k_final<2><<<nb, kBlock, 0, s>>>(c, g, scal, R, rho, ux, uy, uz, T, pmass, guard,
                                         fused);
}

void launch_commit_collide2(const DevCloud &c, double *g, double *gt, double dt,
                            double tau, double R, double *rho, double *ux, double *uy,
                            double *T, double *limflag, double *pnew, double *pmass,
                            hipStream_t s)
{
    const int nb = (c.N + kBlock / kWave - 1) / (kBlock / kWave);
    // rows of up to 256 nodes (Nv <= 16) stay in registers
    const int u = (c.nodes + kWave - 1) / kWave;
    if (u == 1)
        k_commit_collide2<1><<<nb, kBlock, 0, s>>>(c, g, gt, dt, tau, R, rho, ux, uy, T, limflag,
                                                   pnew, pmass);
    else if (u == 2)
        k_commit_collide2<2><<<nb, kBlock, 0, s>>>(c, g, gt, dt, tau, R, rho, ux, uy, T, limflag,
                                                   pnew, pmass);
    else if (u <= 4)
        k_commit_collide2<4><<<nb, kBlock, 0, s>>>(c, g, gt, dt, tau, R, rho, ux, uy, T, limflag,
                                                   pnew, pmass);
    else
        k_commit_collide2<0><<<nb, kBlock, 0, s>>>(c, g, gt, dt, tau, R, rho, ux, uy, T, limflag,
                                                   pnew, pmass);
}

void launch_commit_collide3(const DevCloud &c, double *g, double *gt, double dt,
                            double tau, double R, const double *rho, double *rho_wall, double *ux,
                            double *uy, double *uz, double *T, double *limflag, double *pnew,
                            double *pmass, hipStream_t s)
{
    const int nb = (c.N + kBlock / kWave - 1) / (kBlock / kWave);
    const unsigned n1 = (unsigned)c.Nv, n2 = n1 * n1;
    const unsigned mg1 = (unsigned)((0x100000000ull + n1 - 1) / n1),
                   mg2 = (unsigned)((0x100000000ull + n2 - 1) / n2);
    auto go = [&](auto kernel) {
        kernel<<<nb, kBlock, 0, s>>>(c, g, gt, mg1, mg2, dt, tau, R, rho, rho_wall, ux, uy, uz, T,
                                     limflag, pnew, pmass);
    };
    // rows of up to 1,024 nodes (Nv <= 10) stay in registers
    const int u = (c.nodes + kWave - 1) / kWave;
    if (u <= 4) go(k_commit_collide3<4>);
    else if (u <= 8) go(k_commit_collide3<8>);
    else if (u <= 16) go(k_commit_collide3<16>);
    else go(k_commit_collide3<0>);
}

void launch_mood_check(const DevCloud &c, double *gt, const double *rho, int *mood,
                       double *limflag, hipStream_t s)
{
    if (c.dim == 3) k_mood_check<3><<<c.N, kBlock, 0, s>>>(c, gt, rho, mood, limflag);
    else k_mood_check<2><<<c.N, kBlock, 0, s>>>(c, gt, rho, mood, limflag);
}

void launch_mood_commit(const DevCloud &c, double *g, double *gt, const int *mood,
                        double *limflag, double *pmass, hipStream_t s)
{
    if (c.dim == 3) k_mood_commit<3><<<c.N, kBlock, 0, s>>>(c, g, gt, mood, limflag, pmass);
    else k_mood_commit<2><<<c.N, kBlock, 0, s>>>(c, g, gt, mood, limflag, pmass);
}

void launch_pad_check(const DevCloud &c, const double *g, const double *rho, const double *T,
                      double *limflag, int *fail, hipStream_t s)
{
    k_pad_check<<<c.N, kBlock, 0, s>>>(c, g, rho, T, limflag, fail);
}

}  // namespace ab
