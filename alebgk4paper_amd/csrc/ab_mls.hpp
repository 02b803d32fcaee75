// ab_mls.hpp -- assembly and solve of one MLS system (device helpers of the
// FP64 transport kernels).
#pragma once
#include "ab_device.hpp"

namespace ab {

// Index of the monomial x^a y^b z^c (degree <= 4) in the order of mono3_add.
__host__ __device__ constexpr int mono3(int a, int b, int c)
{
    constexpr int e[35][3] = {
        {0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {2, 0, 0}, {0, 2, 0}, {0, 0, 2},
        {1, 1, 0}, {1, 0, 1}, {0, 1, 1}, {3, 0, 0}, {2, 1, 0}, {2, 0, 1}, {1, 2, 0},
        {1, 1, 1}, {1, 0, 2}, {0, 3, 0}, {0, 2, 1}, {0, 1, 2}, {0, 0, 3}, {4, 0, 0},
        {3, 1, 0}, {3, 0, 1}, {2, 2, 0}, {2, 1, 1}, {2, 0, 2}, {1, 3, 0}, {1, 2, 1},
        {1, 1, 2}, {1, 0, 3}, {0, 4, 0}, {0, 3, 1}, {0, 2, 2}, {0, 1, 3}, {0, 0, 4}};
    for (int k = 0; k < 35; ++k)
        if (e[k][0] == a && e[k][1] == b && e[k][2] == c) return k;
    return -1;
}

// Exponents of the 3-D basis (MLSTransport/MLSBasis.hpp:180-194): 1, x, y, z,
// x^2, y^2, z^2, xy, xz, yz. The first ten monomials are the same functions in
// the same order.
__host__ __device__ constexpr int bexp3(int p, int axis)
{
    constexpr int e[10][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {2, 0, 0},
                              {0, 2, 0}, {0, 0, 2}, {1, 1, 0}, {1, 0, 1}, {0, 1, 1}};
    return e[p][axis];
}

__host__ __device__ constexpr int pair3(int p, int q)
{
    return mono3(bexp3(p, 0) + bexp3(q, 0), bexp3(p, 1) + bexp3(q, 1), bexp3(p, 2) + bexp3(q, 2));
}

// 2-D: monomials up to degree 4, basis 1, x, y, x^2, xy, y^2.
__host__ __device__ constexpr int mono2(int a, int b)
{
    constexpr int e[15][2] = {{0, 0}, {1, 0}, {0, 1}, {2, 0}, {1, 1}, {0, 2}, {3, 0}, {2, 1},
                              {1, 2}, {0, 3}, {4, 0}, {3, 1}, {2, 2}, {1, 3}, {0, 4}};
    for (int k = 0; k < 15; ++k)
        if (e[k][0] == a && e[k][1] == b) return k;
    return -1;
}

__host__ __device__ constexpr int bexp2(int p, int axis)
{
    constexpr int e[6][2] = {{0, 0}, {1, 0}, {0, 1}, {2, 0}, {1, 1}, {0, 2}};
    return e[p][axis];
}

__host__ __device__ constexpr int pair2(int p, int q)
{
    return mono2(bexp2(p, 0) + bexp2(q, 0), bexp2(p, 1) + bexp2(q, 1));
}

// The upper triangle (FULL: all entries) of A from the monomial sums, with the
// indices as template constants (a run-time index would put m in memory).
template <int DIM, int P, bool FULL, int E = 0, int NM>
__device__ __forceinline__ void fill_matrix(const double (&m)[NM], double (&A)[P * P])
{
    if constexpr (E < P * P)
    {
        constexpr int p = E / P, q = E % P;
        constexpr int k = DIM == 3 ? pair3(p, q) : pair2(p, q);
        if constexpr (FULL || q >= p) A[E] = m[k];
        fill_matrix<DIM, P, FULL, E + 1>(m, A);
    }
}

// Adds one neighbour of weight w at (x, y, z) (scaled by the support radius,
// from the foot point) with value g: the monomial sums m and, with RHS, the
// right-hand side r of P basis functions.
template <int P, bool RHS = true>
__device__ __forceinline__ void mono3_add(double w, double x, double y, double z, double g,
                                          double (&m)[P == 10 ? 35 : 10], double (&r)[P])
{
    const double wx = w * x, wy = w * y, wz = w * z;
    m[0] += w; m[1] += wx; m[2] += wy; m[3] += wz;
    if constexpr (RHS) { r[0] += w * g; r[1] += wx * g; r[2] += wy * g; r[3] += wz * g; }
    if constexpr (P < 10)
    {
        m[4] += wx * x; m[5] += wy * y; m[6] += wz * z;
        m[7] += wx * y; m[8] += wx * z; m[9] += wy * z;
    }
    else
    {
        const double xx = wx * x, yy = wy * y, zz = wz * z, xy = wx * y, xz = wx * z, yz = wy * z;
        m[4] += xx; m[5] += yy; m[6] += zz; m[7] += xy; m[8] += xz; m[9] += yz;
        if constexpr (RHS)
        {
            r[4] += xx * g; r[5] += yy * g; r[6] += zz * g;
            r[7] += xy * g; r[8] += xz * g; r[9] += yz * g;
        }
        const double x3 = xx * x, x2y = xx * y, x2z = xx * z, xy2 = xy * y, xyz = xy * z,
                     xz2 = xz * z, y3 = yy * y, y2z = yy * z, yz2 = yz * z, z3 = zz * z;
        m[10] += x3; m[11] += x2y; m[12] += x2z; m[13] += xy2; m[14] += xyz;
        m[15] += xz2; m[16] += y3; m[17] += y2z; m[18] += yz2; m[19] += z3;
        m[20] += x3 * x; m[21] += x3 * y; m[22] += x3 * z; m[23] += x2y * y; m[24] += x2y * z;
        m[25] += x2z * z; m[26] += xy2 * y; m[27] += xy2 * z; m[28] += xyz * z; m[29] += xz2 * z;
        m[30] += y3 * y; m[31] += y3 * z; m[32] += y2z * z; m[33] += yz2 * z; m[34] += z3 * z;
    }
}

// Symmetric elimination of the upper triangle A (P x P, row-major) with the
// right-hand side r, then the back substitution: r becomes the solution
// (its constant term r[0] is the value at the foot point). The pivots are those of the reference's Cholesky
// factorisation, squared; false when one is not above tol times the largest
// diagonal entry (the reference's relative tolerance).
template <int P>
__device__ __forceinline__ bool solve_spd(double (&A)[P * P], double (&r)[P], double tol)
{
    double dmax = 0.0;
#pragma unroll
    for (int k = 0; k < P; ++k) dmax = fmax(dmax, A[k * P + k]);
    bool ok = dmax > 0.0;
    double inv[P];
#pragma unroll
    for (int k = 0; k < P; ++k)
    {
        const double d = A[k * P + k];
        ok = ok && (d > tol * dmax);
        inv[k] = 1.0 / (ok ? d : 1.0);
#pragma unroll
        for (int i = k + 1; i < P; ++i)
        {
            const double f = A[k * P + i] * inv[k];
#pragma unroll
            for (int q = i; q < P; ++q) A[i * P + q] -= f * A[k * P + q];
            r[i] -= f * r[k];
        }
    }
#pragma unroll
    for (int k = P - 1; k >= 0; --k)
    {
        double v = r[k];
#pragma unroll
        for (int i = k + 1; i < P; ++i) v -= A[k * P + i] * r[i];
        r[k] = v * inv[k];
    }
    return ok;
}

}  // namespace ab
