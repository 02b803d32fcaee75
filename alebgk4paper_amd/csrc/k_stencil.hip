// k_stencil.hip -- the 3-D MLS transport of the FP64 formulation where many
// particles have congruent stencils.
//
// The value at the foot point is linear in g: gt[i,v] = sum_o C[o,v] g[i+o,v],
// with C fixed by the stencil's geometry, the wall state and dt. Particles
// whose neighbours sit at the same displacements (the lattice away from
// bodies) share C, so the step assembles and factorises the normal equations
// once per (distinct stencil, node) and applies them to every particle of the
// class. What is in no class (around a body, after a merge, on a jittered
// cloud) goes through k_transport3d, particle by particle.
//
// A class is found from the lists alone, on the device, whenever positions,
// lists or wall state changed (stencil_prepare):
//   k_st_class  one wave per particle: the neighbours on the 81 lattice offsets
//               |o|^2 <= 6, filling a box of them completely, with the ids of
//               every x row consecutive. The key is the box and the boundary
//               flag.
//   k_st_slots  a coefficient slot for every key with enough members.
//   k_st_check  one wave per particle: displacements (to 1e-13 of the support
//               radius, rounding of lattice positions) and, bit for bit, wall
//               normal, wall velocity and mesh velocity as the key's first
//               particle has them; else the particle leaves the class.
//   k_st_follow, k_st_cut, k_st_emit, k_st_scan  runs of consecutive particles of one
//               class whose rows all move by one with the particle, cut into
//               pieces of up to 8 (k_st_cut), four pieces one above the other
//               in y joined to a patch, sorted into bins for the apply's
//               locality; the rest into the lists of k_transport3d.
// Every step: k_stencil_coef, then k_apply_runs.
//
// What bounds the apply is the L2-to-CU traffic (about 12 TB/s on this chip,
// whatever the kernel), so loads per output are what counts. g is N x gstride
// FP64, particle-major: 64 nodes of one particle are one 512-byte load. A run
// of 8 particles along x reads each of its 21 stencil rows once for up to 5 x 8
// products, and four runs one above the other share rows and coefficients: 36
// rows of 10 or 12 loads and 81 coefficients for 32 outputs, 16 loads per
// output against 39 for a single run of 8 and 162 particle by particle.
// 40^3 / Nv 10 quadratic, ms per transport: 25.5 with the full normal matrix
// and 13.6 with the distinct sums per particle; shared, in runs of 12: 2.5 in
// arbitrary order, 2.2 in bins; in patches 1.1, plus 0.04 for the coefficients
// and 0.05 for the 64 corner particles that no other particle is congruent to.
#include "ab_device.hpp"
#include "ab_internal.hpp"
#include "ab_mls.hpp"

#include <algorithm>
#include <climits>
#include <utility>

namespace ab {

namespace {

constexpr int kOff = 81;              // stencil offsets, the particle itself included
constexpr int kRows = 21;             // (oy, oz) rows of 5 or 3 x offsets
constexpr int kRowPad = 24;           // ids per particle in the row table
constexpr int kBoxes = 729;           // extents 0..2 to each of the six sides
constexpr int kKeys = 2 * kBoxes;     // box and boundary flag
constexpr int kCoefRows = kOff + 1;   // coefficients, then the degeneracy flag
constexpr int kRun = 8;               // longest piece of a run
constexpr int kPatch = 4;             // runs of a patch
constexpr int kItem = 8;              // ints per item: length, runs, their first particles
// A class of fewer members is not worth its own factorisation.
constexpr int kMinMembers = 4;

// Counters of the classification (ctx->st_n).
// N_TICKET: the next item of each XCD's share of the apply.
enum { N_SLOT = 0, N_RUN, N_INT, N_BND, N_TICKET = 8, N_COUNT = 16 };

struct Row { int oy, oz, d, o0; };

struct RowTab
{
    Row r[kRows];
    int of[25];                       // row of (oy + 2) + 5 (oz + 2), or -1
    static constexpr RowTab make()
    {
        RowTab t{};
        int n = 0, o0 = 0;
        for (int oz = -2; oz <= 2; ++oz)
            for (int oy = -2; oy <= 2; ++oy)
            {
                const int q = oy * oy + oz * oz, d = q <= 2 ? 2 : (q <= 5 ? 1 : -1);
                t.of[(oy + 2) + 5 * (oz + 2)] = d < 0 ? -1 : n;
                if (d < 0) continue;
                t.r[n++] = Row{oy, oz, d, o0};
                o0 += 2 * d + 1;
            }
        return t;
    }
};
constexpr RowTab kRowTab = RowTab::make();
static_assert(kRowTab.r[kRows - 1].o0 + 2 * kRowTab.r[kRows - 1].d + 1 == kOff, "stencil rows");
__host__ __device__ constexpr int row_of(int oy, int oz)
{
    return oy < -2 || oy > 2 || oz < -2 || oz > 2 ? -1 : kRowTab.of[(oy + 2) + 5 * (oz + 2)];
}
constexpr int kSelfRow = kRowTab.of[12];
constexpr int kSelf = kRowTab.r[kSelfRow].o0 + 2;

// Offset o of the table: its row and (ox, oy, oz).
struct Tap { int row, ox, oy, oz; };
struct TapTab
{
    Tap t[kOff];
    static constexpr TapTab make()
    {
        TapTab r{};
        for (int k = 0; k < kRows; ++k)
            for (int j = 0; j <= 2 * kRowTab.r[k].d; ++j)
                r.t[kRowTab.r[k].o0 + j] = Tap{k, j - kRowTab.r[k].d, kRowTab.r[k].oy, kRowTab.r[k].oz};
        return r;
    }
};
__constant__ constexpr TapTab kTaps = TapTab::make();
__constant__ constexpr RowTab kRowsDev = RowTab::make();

// Whether the box of key k (extents lo, hi per axis) holds the offset.
__device__ __forceinline__ bool in_box(int k, int ox, int oy, int oz)
{
    k %= kBoxes;
    const int ex = k % 9, ey = (k / 9) % 9, ez = k / 81;
    return ox >= -(ex / 3) && ox <= ex % 3 && oy >= -(ey / 3) && oy <= ey % 3 &&
           oz >= -(ez / 3) && oz <= ez % 3;
}

__global__ void k_st_init(int *rep, int *cnt, int *n, int nbin, int *bin)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nbin) bin[k] = 0;
    if (k < kKeys) { rep[k] = INT_MAX; cnt[k] = 0; }
    if (k < N_COUNT) n[k] = 0;
}

__global__ __launch_bounds__(kBlock) void k_st_class(DevCloud c, double isx, double isy, double isz,
                                                     int *__restrict__ key, int *__restrict__ rb,
                                                     int *rep, int *cnt)
{
    __shared__ int srow[kBlock / kWave][kRowPad];
    __shared__ unsigned smask[kBlock / kWave][3];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int i = blockIdx.x * (kBlock / kWave) + w;
    if (i >= c.N) return;                              // whole wave
    const int nn = c.nneigh[i];
    if (lane < kRowPad) srow[w][lane] = lane == kSelfRow ? i : -1;
    if (lane < 3) smask[w][lane] = 0u;
    wave_lds_sync();
    const double xi = c.x[i], yi = c.y[i], zi = c.z[i];
    bool ok = nn < kOff;
    int j[2] = {0, 0}, ox[2] = {0, 0}, row[2] = {-1, -1};
#pragma unroll
    for (int q = 0; q < 2; ++q)
    {
        const int t = lane + q * kWave;
        if (!ok || t >= nn) continue;
        j[q] = c.neigh[(size_t)i * AB_MAX_NEIGH + t];
        const double dx = (c.x[j[q]] - xi) * isx, dy = (c.y[j[q]] - yi) * isy,
                     dz = (c.z[j[q]] - zi) * isz;
        const double rx = rint(dx), ry = rint(dy), rz = rint(dz);
        // (near a lattice offset at all; how near is k_st_check's question)
        bool in = fabs(dx - rx) < 1e-3 && fabs(dy - ry) < 1e-3 && fabs(dz - rz) < 1e-3 &&
                  fabs(rx) <= 2.0 && fabs(ry) <= 2.0 && fabs(rz) <= 2.0;
        if (in)
        {
            ox[q] = (int)rx;
            row[q] = kRowsDev.of[((int)ry + 2) + 5 * ((int)rz + 2)];
            in = row[q] >= 0 && abs(ox[q]) <= kRowsDev.r[row[q]].d;
        }
        const int o = in ? kRowsDev.r[row[q]].o0 + ox[q] + kRowsDev.r[row[q]].d : kSelf;
        if (!in || o == kSelf) { ok = false; row[q] = -1; continue; }
        if (ox[q] == 0) srow[w][row[q]] = j[q];
        atomicOr(&smask[w][o >> 5], 1u << (o & 31));
    }
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (row[q] >= 0) ok = ok && srow[w][row[q]] >= 0 && j[q] == srow[w][row[q]] + ox[q];
    unsigned m[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) m[q] = smask[w][q];
    // as many offsets as neighbours: none twice
    ok = ok && (int)(__popc(m[0]) + __popc(m[1]) + __popc(m[2])) == nn;
    m[kSelf >> 5] |= 1u << (kSelf & 31);
    auto has = [&](int o) { return (m[o >> 5] >> (o & 31)) & 1u; };
    auto tap = [&](int x, int y, int z) {
        const int r = kRowTab.of[(y + 2) + 5 * (z + 2)];
        return kRowTab.r[r].o0 + x + kRowTab.r[r].d;
    };
    auto ext = [&](int x, int y, int z) {
        return has(tap(x, y, z)) ? (has(tap(2 * x, 2 * y, 2 * z)) ? 2 : 1) : 0;
    };
    const int ex = 3 * ext(-1, 0, 0) + ext(1, 0, 0), ey = 3 * ext(0, -1, 0) + ext(0, 1, 0),
              ez = 3 * ext(0, 0, -1) + ext(0, 0, 1);
    const int k = ex + 9 * (ey + 9 * ez) + (c.bnd[i] ? kBoxes : 0);
#pragma unroll
    for (int q = 0; q < 2; ++q)
    {
        const int o = lane + q * kWave;
        if (o < kOff)
        {
            const Tap t = kTaps.t[o];
            ok = ok && in_box(k, t.ox, t.oy, t.oz) == (bool)has(o);
        }
    }
    ok = __all(ok);
    // an absent row reads the particle's own (its coefficients are zero)
    if (lane < kRowPad) rb[(size_t)i * kRowPad + lane] = lane < kRows && srow[w][lane] >= 0 ? srow[w][lane] : i;
    if (lane == 0)
    {
        key[i] = ok ? k : -1;
        // the plain reads spare most of the atomics on the one interior key;
        // a stale value only costs one more
        if (ok && rep[k] > i) atomicMin(&rep[k], i);
        if (ok && cnt[k] < kMinMembers) atomicAdd(&cnt[k], 1);
    }
}

// Slots in key order, one wave.
__global__ __launch_bounds__(kWave) void k_st_slots(const int *__restrict__ cnt, int *__restrict__ slot,
                                                    int *__restrict__ skey, int maxslot, int *n)
{
    const int lane = threadIdx.x;
    int used = 0;
    for (int k0 = 0; k0 < kKeys; k0 += kWave)
    {
        const int k = k0 + lane;
        const bool want = k < kKeys && cnt[k] >= kMinMembers;
        const unsigned long long b = __ballot(want);
        const int at = used + __popcll(b & ((1ull << lane) - 1ull));
        if (k < kKeys) slot[k] = want && at < maxslot ? at : -1;
        if (want && at < maxslot) skey[at] = k;
        used += __popcll(b);
    }
    if (lane == 0) n[N_SLOT] = min(used, maxslot);
}

__global__ __launch_bounds__(kBlock) void k_st_check(DevCloud c, double tol, int *key,
                                                     const int *__restrict__ rb,
                                                     const int *__restrict__ rep,
                                                     const int *__restrict__ slot)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int i = blockIdx.x * (kBlock / kWave) + (int)(threadIdx.x / kWave);
    if (i >= c.N) return;                              // whole wave
    const int k = key[i];
    if (k < 0) return;
    bool ok = slot[k] >= 0;
    const int r = rep[k];
    if (ok && r != i)
    {
#pragma unroll
        for (int q = 0; q < 2; ++q)
        {
            const int o = lane + q * kWave;
            if (o >= kOff) continue;
            const Tap t = kTaps.t[o];
            if (!in_box(k, t.ox, t.oy, t.oz)) continue;
            const int a = rb[(size_t)i * kRowPad + t.row] + t.ox;
            const int b = rb[(size_t)r * kRowPad + t.row] + t.ox;
            ok = ok && fabs((c.x[a] - c.x[i]) - (c.x[b] - c.x[r])) <= tol &&
                 fabs((c.y[a] - c.y[i]) - (c.y[b] - c.y[r])) <= tol &&
                 fabs((c.z[a] - c.z[i]) - (c.z[b] - c.z[r])) <= tol;
        }
        ok = ok && c.mvx[i] == c.mvx[r] && c.mvy[i] == c.mvy[r] && c.mvz[i] == c.mvz[r];
        if (c.bnd[i])
            ok = ok && c.wnx[i] == c.wnx[r] && c.wny[i] == c.wny[r] && c.wnz[i] == c.wnz[r] &&
                 c.wux[i] == c.wux[r] && c.wuy[i] == c.wuy[r] && c.wuz[i] == c.wuz[r];
    }
    if (!__all(ok) && lane == 0) key[i] = -1;
}

// Whether particle i continues the run of particle i - 1.
__global__ void k_st_follow(int N, const int *__restrict__ key, const int *__restrict__ rb,
                            unsigned char *__restrict__ follow, unsigned char *__restrict__ plen)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    bool f = i > 0 && key[i] >= 0 && key[i] == key[i - 1];
    if (f)
    {
        const int *a = rb + (size_t)(i - 1) * kRowPad, *b = a + kRowPad;
        for (int r = 0; r < kRows; ++r) f = f && b[r] == a[r] + 1;
    }
    follow[i] = f;
    plen[i] = 0;
}

// plen: the length of the piece that starts at particle i, or 0.
__global__ void k_st_cut(int N, const int *__restrict__ key, const unsigned char *__restrict__ follow,
                         unsigned char *__restrict__ plen)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N || key[i] < 0 || follow[i]) return;
    int len = 1;
    while (i + len < N && follow[i + len]) ++len;
    for (int a = 0; a < len; a += kRun) plen[i + a] = (unsigned char)min(kRun, len - a);
}

// The piece one lattice row up (+y) from the piece at i that can share its
// loads: same class and length, and every stencil row of it that the table of
// i's run has one row further up (oy + 1) is that row. A patch reads row (y, oz)
// through the first of its runs whose 21 rows reach it, so a box that ends at
// oy = 1 forms no patch: there row oy = 1 of a later run would be read through
// row oy = 2 of an earlier one, which has none. -1: none.
__device__ __forceinline__ int piece_up(int i, const int *__restrict__ key, const int *__restrict__ rb,
                                        const unsigned char *__restrict__ plen)
{
    const int *a = rb + (size_t)i * kRowPad;
    const int t = a[row_of(1, 0)], k = key[i];
    if (t == i || key[t] != k || plen[t] != plen[i]) return -1;
    const int *b = rb + (size_t)t * kRowPad;
    bool ok = true;
    for (int r = 0; r < kRows; ++r)
    {
        const Row q = kRowsDev.r[r];
        const int up = q.oy < 2 ? kRowsDev.of[(q.oy + 3) + 5 * (q.oz + 2)] : -1;
        if (up >= 0 && in_box(k, 0, q.oy, q.oz))
            ok = ok && in_box(k, 0, q.oy + 1, q.oz) && b[r] == a[up];
    }
    return ok ? t : -1;
}

// The bin of a run in the apply's order: strips of kStrip lattice rows in y,
// and within a strip plane by plane in z. The runs in flight on an XCD (about
// 500 waves) then read a window of a dozen rows by a dozen planes, 3 MB of one
// chunk's values at 40 particles a row, and stay in its 4 MB L2.
constexpr int kStrip = 8;

struct Bins { double y0, z0, isy, isz; int ny, nz; };

__device__ __forceinline__ int bin_of(const DevCloud &c, const Bins &b, int i)
{
    const double y = (c.y[i] - b.y0) * b.isy / kStrip, z = rint((c.z[i] - b.z0) * b.isz);
    const int iy = (int)fmin(fmax(y, 0.0), b.ny - 1.0), iz = (int)fmin(fmax(z, 0.0), b.nz - 1.0);
    return iy * b.nz + iz;
}

// The place in its patch that a piece of key k asks for: its lattice row counted
// from the key's first particle, which keeps lattice rows 2, 6, 10, ... first
// and, wherever the lattice lies, y differences near whole spacings.
__device__ __forceinline__ int patch_place(const DevCloud &c, const Bins &bins, int i, int r)
{
    return (int)rint((c.y[i] - c.y[r]) * bins.isy) & (kPatch - 1);
}

// Whether the piece at base is the first of a patch, its pieces into at: places
// 0 .. kPatch - 1 in turn, each linked to the next upwards (piece_up) and
// downwards. So a piece belongs to one patch at most, the one that its own links
// lead down to, and every piece that asks gets the same answer, whatever the
// spacing that the places are counted with.
__device__ __forceinline__ bool patch_at(const DevCloud &c, const Bins &bins, int base,
                                         const int *__restrict__ key, const int *__restrict__ rb,
                                         const int *__restrict__ rep,
                                         const unsigned char *__restrict__ plen, int (&at)[kPatch])
{
    at[0] = base;
    if (key[base] < 0 || !plen[base]) return false;
    const int r = rep[key[base]];
    if (patch_place(c, bins, base, r) != 0) return false;
    for (int q = 1; q < kPatch; ++q)
    {
        const int t = piece_up(at[q - 1], key, rb, plen);
        if (t < 0 || patch_place(c, bins, t, r) != q ||
            rb[(size_t)t * kRowPad + row_of(-1, 0)] != at[q - 1])
            return false;
        at[q] = t;
    }
    return true;
}

// Items: patches of kPatch pieces one above the other in y, where all of them
// are there, else single pieces. Counted per bin (COUNT), then placed from the
// bin's start; the particles of no class into their lists.
template <bool COUNT>
__global__ void k_st_emit(DevCloud c, Bins bins, const int *__restrict__ key,
                          const int *__restrict__ rb, const int *__restrict__ rep,
                          const unsigned char *__restrict__ plen, int *bin,
                          int *__restrict__ item, int *__restrict__ irr_int,
                          int *__restrict__ irr_bnd, int *n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.N) return;
    if (key[i] < 0)
    {
        if (COUNT) return;
        if (c.bnd[i]) irr_bnd[atomicAdd(&n[N_BND], 1)] = i;
        else irr_int[atomicAdd(&n[N_INT], 1)] = i;
        return;
    }
    if (!plen[i]) return;
    const int place = patch_place(c, bins, i, rep[key[i]]);
    int base = i;
    for (int q = 0; q < place; ++q) base = rb[(size_t)base * kRowPad + row_of(-1, 0)];
    int at[kPatch];
    const bool patch = patch_at(c, bins, base, key, rb, rep, plen, at) && at[place] == i;
    if (patch && place) return;                        // its first piece places the patch
    const int k = atomicAdd(&bin[bin_of(c, bins, i)], 1);
    if (COUNT) return;
    int *o = item + (size_t)k * kItem;
    o[0] = plen[i];
    o[1] = patch ? kPatch : 1;
    for (int q = 0; q < kPatch; ++q) o[2 + q] = patch ? at[q] : i;
}

// Exclusive scan of the bin counts in place, one workgroup.
__global__ __launch_bounds__(1024) void k_st_scan(int nbin, int *bin, int *n)
{
    __shared__ int sh[1024];
    const int t = threadIdx.x, per = (nbin + 1023) / 1024;
    const int lo = min(t * per, nbin), hi = min(lo + per, nbin);
    int s = 0;
    for (int k = lo; k < hi; ++k) s += bin[k];
    sh[t] = s;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1)
    {
        const int v = t >= d ? sh[t - d] : 0;
        __syncthreads();
        sh[t] += v;
        __syncthreads();
    }
    int at = sh[t] - s;
    for (int k = lo; k < hi; ++k) { const int v = bin[k]; bin[k] = at; at += v; }
    if (t == 1023) n[N_RUN] = sh[1023];
}

// The coefficients of one class's 64 nodes: the normal equations of the key's
// first particle (the same sums and solve as k_transport3d), q = A^-1 e0, then
// C_o = w_o phi_o . q. The weights w / sum w where a pivot collapses; the
// particle's own value where a wall node is gated or no neighbour has weight.
// An offset that does not enter holds -0.0, one that does never does, so the
// apply can tell them apart. About 6,000 FP64 instructions per node for a
// few dozen classes: 1 % of the step's assembly per particle.
template <int P, bool BND>
__device__ __forceinline__ void coef_nodes(const DevCloud &c, int i, int lin, double dt, double h,
                                           double tol, const double (&se)[kOff][4],
                                           double *__restrict__ out)
{
    const int Nv = c.Nv;
    const double vx = vnode(c.vlo, c.dv, lin % Nv);
    const double vy = vnode(c.vlo, c.dv, (lin / Nv) % Nv);
    const double vz = vnode(c.vlo, c.dv, lin / (Nv * Nv));
    const double ih = 1.0 / h;
    bool own = false;
    if (BND)
        own = wall_cn3(vx, vy, vz, c.wux[i], c.wuy[i], c.wuz[i], c.wnx[i], c.wny[i],
                       c.wnz[i]) >= 0.0;
    const double ox = (vx - c.mvx[i]) * dt * ih, oy = (vy - c.mvy[i]) * dt * ih,
                 oz = (vz - c.mvz[i]) * dt * ih;
    constexpr int NM = P == 10 ? 35 : 10;
    double m[NM], r[P];
#pragma unroll
    for (int q = 0; q < NM; ++q) m[q] = 0.0;
#pragma unroll
    for (int q = 0; q < P; ++q) r[q] = q == 0 ? 1.0 : 0.0;
    auto weight = [&](int o, double &x, double &y, double &z) {
        x = se[o][0] + ox; y = se[o][1] + oy; z = se[o][2] + oz;
        const double u = fmax(1.0 - (x * x + y * y + z * z), 0.0);
        const double w = u * u;
        return w < 1e-30 ? 0.0 : w;
    };
    for (int o = 0; o < kOff; ++o)
    {
        if (se[o][3] == 0.0) continue;                 // not in the box, or the particle itself
        double x, y, z;
        const double w = weight(o, x, y, z);
        mono3_add<P, false>(w, x, y, z, 0.0, m, r);
    }
    const double sumW = m[0];
    own = own || !(sumW > 0.0);
    double A[P * P];
    fill_matrix<3, P, false>(m, A);
    bool ok = solve_spd<P>(A, r, tol);
#pragma unroll
    for (int q = 0; q < P; ++q) ok = ok && isfinite(r[q]);
    for (int o = 0; o < kOff; ++o)
    {
        double cm = -0.0;
        if (se[o][3] != 0.0)
        {
            double x, y, z;
            const double w = weight(o, x, y, z);
            double f = r[0] + r[1] * x + r[2] * y + r[3] * z;
            if constexpr (P == 10)
                f += r[4] * (x * x) + r[5] * (y * y) + r[6] * (z * z) + r[7] * (x * y) +
                     r[8] * (x * z) + r[9] * (y * z);
            const double v = ok ? w * f : w / sumW;
            if (w > 0.0 && !own) cm = v == 0.0 ? 0.0 : v;
        }
        else if (o == kSelf && own) cm = 1.0;
        out[(size_t)o * kWave] = cm;
    }
    out[(size_t)kOff * kWave] = ok || own ? 0.0 : 1.0;
}

__global__ __launch_bounds__(kWave) void k_stencil_coef(DevCloud c, double dt, double h, double tol,
                                                        int order, int *n,
                                                        const int *__restrict__ skey,
                                                        const int *__restrict__ rep,
                                                        const int *__restrict__ rb, int nchunk,
                                                        double *__restrict__ coef)
{
    __shared__ double se[kOff][4];
    const int slot = blockIdx.y, chunk = blockIdx.x;
    if (slot + chunk == 0 && threadIdx.x < 8) n[N_TICKET + threadIdx.x] = 0;   // for the apply
    if (slot >= n[N_SLOT]) return;
    const int k = skey[slot], i = rep[k];
    const double ih = 1.0 / h;
    for (int o = threadIdx.x; o < kOff; o += kWave)
    {
        const Tap t = kTaps.t[o];
        const bool in = o != kSelf && in_box(k, t.ox, t.oy, t.oz);
        const int j = in ? rb[(size_t)i * kRowPad + t.row] + t.ox : i;
        se[o][0] = (c.x[j] - c.x[i]) * ih;
        se[o][1] = (c.y[j] - c.y[i]) * ih;
        se[o][2] = (c.z[j] - c.z[i]) * ih;
        se[o][3] = in ? 1.0 : 0.0;
    }
    __syncthreads();
    // the last chunk's lanes past the row repeat its last node
    const int lin = min(chunk * kWave + (int)threadIdx.x, c.nodes - 1);
    double *out = coef + ((size_t)slot * nchunk + chunk) * kCoefRows * kWave + threadIdx.x;
    if (c.bnd[i]) coef_nodes<4, true>(c, i, lin, dt, h, tol, se, out);
    else if (order >= 2) coef_nodes<10, false>(c, i, lin, dt, h, tol, se, out);
    else coef_nodes<4, false>(c, i, lin, dt, h, tol, se, out);
}

struct RunArgs
{
    const double *g;
    double *gt;
    const double *coef;
    const int *rb;
    double dt, h;
    int clamp;
    int *mlsflag;
    double *mlsovr;
};

__device__ __forceinline__ bool enters(double cm)
{
    return (unsigned)(__builtin_bit_cast(unsigned long long, cm) >> 32) != 0x80000000u;
}

// One output the long way: only the offsets that enter, and the Shepard
// average where the value is not finite (a value outside the support must not
// enter, also if it is not finite; 0 x inf would).
__device__ __forceinline__ double output_checked(const DevCloud &c, const double *g, const double *cf,
                                              const int *rb, double dt, double h, int i, int lin,
                                              int voff, double &gmin, double &gmax, bool &bad)
{
    const int Nv = c.Nv;
    const size_t gs = (size_t)c.gstride;
    const double ih = 1.0 / h;
    const double ox = (vnode(c.vlo, c.dv, lin % Nv) - c.mvx[i]) * dt * ih;
    const double oy = (vnode(c.vlo, c.dv, (lin / Nv) % Nv) - c.mvy[i]) * dt * ih;
    const double oz = (vnode(c.vlo, c.dv, lin / (Nv * Nv)) - c.mvz[i]) * dt * ih;
    double acc = 0.0, sw = 0.0, swg = 0.0;
    gmin = 1e300;
    gmax = -1e300;
    bool own = false;
    for (int o = 0; o < kOff; ++o)
    {
        const double cm = cf[(size_t)o * kWave + voff];
        if (!enters(cm)) continue;
        const Tap t = kTaps.t[o];
        const int j = rb[(size_t)i * kRowPad + t.row] + t.ox;
        const double v = g[(size_t)j * gs + lin];
        if (o == kSelf) { own = true; acc = v; }
        const double x = (c.x[j] - c.x[i]) * ih + ox, y = (c.y[j] - c.y[i]) * ih + oy,
                     z = (c.z[j] - c.z[i]) * ih + oz;
        const double u = fmax(1.0 - (x * x + y * y + z * z), 0.0);
        if (o != kSelf) acc += cm * v;
        sw += u * u;
        swg += u * u * v;
        gmin = fmin(gmin, v);
        gmax = fmax(gmax, v);
    }
    bad = !own && !isfinite(acc);
    return bad ? swg / sw : acc;
}

// Stencil rows of a patch of YN runs, relative to its first run: row (y, oz)
// is read once, R + 2 d values, for every run k that has it at oy = y - k.
template <int YN>
struct Patch
{
    struct R1 { int oz, y, d, k; };                    // k: the first run that has the row
    struct Tab { R1 r[5 * (YN + 4)]; int n; };
    static constexpr Tab make()
    {
        Tab t{};
        int n = 0;
        for (int oz = -2; oz <= 2; ++oz)
            for (int y = -2; y <= YN + 1; ++y)
            {
                int d = 0, k0 = -1;
                for (int k = YN - 1; k >= 0; --k)
                    if (row_of(y - k, oz) >= 0)
                    {
                        k0 = k;
                        const int dk = kRowTab.r[row_of(y - k, oz)].d;
                        d = dk > d ? dk : d;
                    }
                if (k0 >= 0) t.r[n++] = R1{oz, y, d, k0};
            }
        t.n = n;
        return t;
    }
    static constexpr Tab tab = make();
};

struct Wave                                            // what the loads of an item need
{
    const double *gl, *cf;                             // values and coefficients of the chunk
    const int *rb;
    int N, voff, lane;
    size_t gs;
};

// Rows in flight: the loads of row U + D - 1 are issued before the products of
// row U. A patch of full pieces has registers for two rows; the others take three
// (a step of 20^3 / Nv 8, 13^3 / Nv 7, 40^3 / Nv 10: 263, 197, 1690 us with two rows
// everywhere, 260, 194, 1671 with three; four are no faster), but not with the
// neighbours' ranges, which the third row costs registers (40^3 / Nv 10 with
// statistics: 3.90 ms with two, 4.33 with three).
template <int YN, int R, bool DIAG>
constexpr int depth() { return DIAG || (R >= 8 && YN > 1) ? 2 : 3; }

// Where the coefficients of the stencil row at oy are kept until the last run of
// the patch has met it: by oy (the same row of the next plane comes after
// that), or in the ring of a single run.
template <int YN, int R, bool DIAG>
constexpr int coef_at(int U, int oy) { return YN > 1 ? oy + 2 : U % depth<YN, R, DIAG>(); }

// Values of patch row U into v, and into cm the coefficients of the stencil row
// that the first run meets there (the later runs meet it at later rows).
template <int YN, int R, bool DIAG, int U>
__device__ __forceinline__ void patch_load(const Wave &w, const int (&first)[YN], double (&v)[R + 4],
                                           double (&cm)[5][5])
{
    constexpr auto q = Patch<YN>::tab.r[U];
    const int b = w.rb[(size_t)first[q.k] * kRowPad + row_of(q.y - q.k, q.oz)];
#pragma clang loop unroll(full)
    for (int j = 0; j < R + 2 * q.d; ++j)
    {
        // ids past the row's end (taps the box cuts off, outputs past the
        // piece's) stay inside the array; their coefficients or outputs do not count
        const int id = min(max(b - q.d + j, 0), w.N - 1);
        v[j] = (w.gl + (size_t)id * w.gs)[w.voff];
    }
    if constexpr (row_of(q.y, q.oz) >= 0)
    {
        constexpr Row k = kRowTab.r[row_of(q.y, q.oz)];
#pragma clang loop unroll(full)
        for (int j = 0; j <= 2 * k.d; ++j)
            cm[coef_at<YN, R, DIAG>(U, q.y)][j] = (w.cf + (size_t)(k.o0 + j) * kWave)[w.lane];
    }
}

template <int YN, int R, bool DIAG, int U>
__device__ __forceinline__ void patch_step(const Wave &w, const int (&first)[YN],
                                           double (&v)[depth<YN, R, DIAG>()][R + 4],
                                           double (&cm)[5][5], double (&acc)[YN][R], double (&gmin)[DIAG ? R : 1],
                                           double (&gmax)[DIAG ? R : 1])
{
    constexpr auto q = Patch<YN>::tab.r[U];
    constexpr int D = depth<YN, R, DIAG>(), B = U % D;
    if constexpr (U + D - 1 < Patch<YN>::tab.n)
        patch_load<YN, R, DIAG, U + D - 1>(w, first, v[(U + D - 1) % D], cm);
#pragma clang loop unroll(full)
    for (int k = 0; k < YN; ++k)
    {
        const int ro = row_of(q.y - k, q.oz);          // constant once unrolled
        if (ro < 0) continue;
        const int d = kRowTab.r[ro].d;
#pragma clang loop unroll(full)
        for (int j = 0; j <= 4; ++j)
        {
            if (j > 2 * d) continue;
            const double cj = cm[coef_at<YN, R, DIAG>(U, q.y - k)][j];
#pragma clang loop unroll(full)
            for (int r = 0; r < R; ++r) acc[k][r] += cj * v[B][r + j + q.d - d];
            if constexpr (DIAG)
            {
                const bool in = enters(cj);
#pragma clang loop unroll(full)
                for (int r = 0; r < R; ++r)
                {
                    gmin[r] = in ? fmin(gmin[r], v[B][r + j]) : gmin[r];
                    gmax[r] = in ? fmax(gmax[r], v[B][r + j]) : gmax[r];
                }
            }
        }
    }
    // the next row's loads stay ahead of this row's products
#pragma clang loop unroll(full)
    for (int k = 0; k < YN; ++k)
#pragma clang loop unroll(full)
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(acc[k][r])::"memory");
    if constexpr (DIAG)
#pragma clang loop unroll(full)
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(gmin[r]), "+v"(gmax[r])::"memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <int YN, int R, bool DIAG, int... U>
__device__ __forceinline__ void patch_rows(const Wave &w, const int (&first)[YN], double (&acc)[YN][R],
                                           double (&gmin)[DIAG ? R : 1],
                                           double (&gmax)[DIAG ? R : 1],
                                           std::integer_sequence<int, U...>)
{
    constexpr int D = depth<YN, R, DIAG>();
    double v[D][R + 4], cm[5][5];
    patch_load<YN, R, DIAG, 0>(w, first, v[0], cm);
    if constexpr (D > 2) patch_load<YN, R, DIAG, 1>(w, first, v[1], cm);
    (patch_step<YN, R, DIAG, U>(w, first, v, cm, acc, gmin, gmax), ...);
}

// One item's outputs: YN runs of len <= R particles, 64 nodes.
template <int YN, int R, bool DIAG>
__device__ __forceinline__ void apply_item(const DevCloud &c, const RunArgs &a, const double *cf,
                                           const int (&first)[YN], int len, int chunk)
{
    static_assert(!DIAG || YN == 1, "ranges are kept for one run");
    const int lane = threadIdx.x & (kWave - 1);
    const int c0 = chunk * kWave, left = c.nodes - c0;
    const size_t gs = (size_t)c.gstride;
    // lanes past the row repeat its last node
    const Wave w{a.g + c0, cf, a.rb, c.N, min(lane, left - 1), lane, gs};
    double acc[YN][R], gmin[DIAG ? R : 1], gmax[DIAG ? R : 1];
#pragma unroll
    for (int k = 0; k < YN; ++k)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[k][r] = 0.0;
    if constexpr (DIAG)
#pragma unroll
        for (int r = 0; r < R; ++r) { gmin[r] = 1e300; gmax[r] = -1e300; }
    patch_rows<YN, R, DIAG>(w, first, acc, gmin, gmax,
                            std::make_integer_sequence<int, Patch<YN>::tab.n>{});
    double degen = 0.0;
    if constexpr (DIAG) degen = cf[(size_t)kOff * kWave + lane];
    unsigned checked = 0;                              // outputs to be done the long way
    auto finish = [&](int i, double out, double lo, double hi, bool bad) {
        if constexpr (DIAG)
        {
            int flag = bad || degen != 0.0 ? 1 : 0;
            double excess = fmax(fmax(out - hi, lo - out), 0.0);
            const bool over = out < lo || out > hi;
            if (over) flag |= 2;
            if (over && a.clamp) out = fmin(fmax(out, lo), hi);
            if (lane >= left) { flag = 0; excess = 0.0; }
            excess = wave_sum(excess);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) flag |= __shfl_xor(flag, o, kWave);
            if (lane == 0 && flag) atomicOr(&a.mlsflag[i], flag);
            if (lane == 0 && excess > 0.0) atomicAdd(&a.mlsovr[i], excess * c.dv * c.dv * c.dv);
        }
        if (lane < left) a.gt[(size_t)i * gs + c0 + lane] = out;
    };
#pragma unroll
    for (int k = 0; k < YN; ++k)
#pragma unroll
        for (int r = 0; r < R; ++r)
        {
            if (r >= len) break;
            if (__any(!isfinite(acc[k][r]))) checked |= 1u << (k * R + r);
            else finish(first[k] + r, acc[k][r], DIAG ? gmin[DIAG ? r : 0] : 0.0,
                        DIAG ? gmax[DIAG ? r : 0] : 0.0, false);
        }
    while (checked)
    {
        const int b = __builtin_ctz(checked), k = b / R;
        checked &= checked - 1;
        int i = first[0];
#pragma unroll
        for (int q = 1; q < YN; ++q) i = q == k ? first[q] : i;
        i += b - k * R;
        double lo, hi;
        bool bad;
        const double out = output_checked(c, a.g, cf, a.rb, a.dt, a.h, i, c0 + w.voff, lane, lo,
                                          hi, bad);
        finish(i, out, lo, hi, bad);
    }
}

// Items are (chunk of 64 nodes, run), the runs of one chunk one after another.
// Each XCD takes a contiguous eighth of them and its waves draw the next item
// from a counter, so the items in flight on it stay neighbours, whatever the
// waves' pace, and share their rows in its L2. (With a fixed stride per wave
// the waves drift apart: 51 % of the requests missed the L2 instead of 10 %.) Every wave ends
// when its share's counter passes the share's end.
template <bool DIAG>
__global__ __launch_bounds__(kBlock, DIAG ? 2 : 3) void k_apply_runs(DevCloud c, RunArgs a, int *n,
                                                       const int *__restrict__ item,
                                                       const int *__restrict__ key,
                                                       const int *__restrict__ slot, int nchunk)
{
    const int nrun = n[N_RUN];
    const int total = nrun * nchunk;
    const int xcd = blockIdx.x & 7;
    const int t0 = (int)((long long)total * xcd / 8), t1 = (int)((long long)total * (xcd + 1) / 8);
    auto draw = [&]() {
        int t = 0;
        if ((threadIdx.x & (kWave - 1)) == 0) t = atomicAdd(&n[N_TICKET + xcd], 1);
        return t0 + __builtin_amdgcn_readfirstlane(t);
    };
    for (int t = draw(); t < t1; t = draw())
    {
        const int chunk = t / nrun;
        const int *it = item + (size_t)(t - chunk * nrun) * kItem;
        const int len = it[0];
        const double *cf = a.coef + ((size_t)slot[key[it[2]]] * nchunk + chunk) * kCoefRows * kWave;
        if constexpr (DIAG)
        {
            // four outputs at a time: the ranges would not fit the registers
            // of a patch (same sums, same bits)
            for (int k = 0; k < it[1]; ++k)
                for (int p = 0; p < len; p += 4)
                {
                    const int first[1] = {it[2 + k] + p};
                    apply_item<1, 4, true>(c, a, cf, first, min(4, len - p), chunk);
                }
        }
        else if (it[1] == kPatch)
        {
            const int first[kPatch] = {it[2], it[3], it[4], it[5]};
            if (len > 4) apply_item<kPatch, 8, false>(c, a, cf, first, len, chunk);
            else if (len > 1) apply_item<kPatch, 4, false>(c, a, cf, first, len, chunk);
            else apply_item<kPatch, 1, false>(c, a, cf, first, len, chunk);
        }
        else
        {
            const int first[1] = {it[2]};
            if (len > 2) apply_item<1, 8, false>(c, a, cf, first, len, chunk);
            else apply_item<1, 2, false>(c, a, cf, first, len, chunk);
        }
    }
}

template <typename T>
bool dev(T **p, size_t n) { return hipMalloc((void **)p, n * sizeof(T)) == hipSuccess; }

}  // namespace

void stencil_free(ab_ctx *c)
{
    void *p[] = {c->st_key, c->st_rb, c->st_rep, c->st_cnt, c->st_slot, c->st_skey, c->st_n,
                 c->st_run, c->st_int, c->st_bnd, c->st_follow, c->st_coef, c->st_bin};
    for (void *q : p) if (q) (void)hipFree(q);
    c->st_key = c->st_rb = c->st_rep = c->st_cnt = c->st_slot = c->st_skey = c->st_n = nullptr;
    c->st_run = c->st_int = c->st_bnd = c->st_bin = nullptr;
    c->st_follow = nullptr;
    c->st_coef = nullptr;
    c->st_cap = 0;
    c->st_valid = false;
}

// The shared path has a floor of about 150 us (the coefficients' chain of dependent
// FP64 operations, the longest items, the corner particles), the per-particle
// path takes 15 us and 0.28 us per 1,000 interior quadratic (or 3,300 linear)
// values. They meet at 500,000: us shared / per particle 205 / 116 at 337,000
// (10^3 / Nv 8), 214 / 183 at 418,000 (12^3 / Nv 7), 160 / 231 at 546,000 (13^3 /
// Nv 7), 170 / 304 at 1.04 million (14^3 / Nv 8); linear 152 / 133 at 421,000, 158 /
// 193 at 629,000.
bool stencil_shared(const ab_ctx *c)
{
    const double w = (c->cfg.mls_order >= 2 ? 1.0 : 0.3) * c->n_int + 0.3 * c->n_bnd;
    return c->dim == 3 && w * c->nodes >= 5e5;
}

// Classes, runs and lists of the cloud as it is now, on its stream, without a
// host synchronisation.
int stencil_prepare(ab_ctx *c)
{
    const size_t N = (size_t)c->N;
    const int nchunk = (c->nodes + kWave - 1) / kWave;
    const ab_config &f = c->cfg;
    // the lattice spacing, a guess that the checks do not rely on: voxels are
    // three spacings wide; without a voxel grid the radius is 2.5 of them
    auto inv = [&](double box) { return box != 0.0 ? 3.0 / box : 2.5 / f.radius; };
    Bins bins{f.ybottom, f.zfront, inv(f.vbox), inv(f.wbox),
              std::min(std::max(3 * f.nbvbox / kStrip + 1, 1), 256),
              std::min(std::max(3 * f.nbwbox + 1, 1), 1024)};
    const int nbin = bins.ny * bins.nz;
    if (N >= (size_t)INT_MAX / kItem)
    { c->err = "FP64 transport: too many particles"; return AB_ERR_UNSUPPORTED; }
    // coefficient slots: the 125 classes of a box lattice and some more, but
    // never more memory than g itself takes
    const size_t one = (size_t)nchunk * kCoefRows * kWave;
    auto slots = [&](size_t n) { return (int)std::min<size_t>(160, n * c->gstride / one); };
    if (c->N > c->st_cap)
    {
        // some room for the particles that cloud management adds
        stencil_free(c);
        const size_t cap = N + N / 16, ms = std::max(slots(cap), 1);
        if (!dev(&c->st_key, cap) || !dev(&c->st_rb, cap * kRowPad) || !dev(&c->st_rep, kKeys) ||
            !dev(&c->st_cnt, kKeys) || !dev(&c->st_slot, kKeys) || !dev(&c->st_skey, ms) ||
            !dev(&c->st_n, N_COUNT) || !dev(&c->st_run, cap * kItem) || !dev(&c->st_int, cap) ||
            !dev(&c->st_bnd, cap) || !dev(&c->st_bin, (size_t)nbin) ||
            !dev(&c->st_follow, 2 * cap) || !dev(&c->st_coef, one * ms))
        { c->err = "FP64 transport: device allocation failed"; return AB_ERR_NOMEM; }
        c->st_cap = (int)cap;
    }
    c->st_maxslot = slots(N);          // of this N, whatever the arrays hold
    DevCloud v = c->view();
    hipStream_t s = c->stream;
    const int nw = (c->N + kBlock / kWave - 1) / (kBlock / kWave), nt = (c->N + 255) / 256;
    k_st_init<<<(std::max(kKeys, nbin) + 255) / 256, 256, 0, s>>>(c->st_rep, c->st_cnt, c->st_n, nbin,
                                                                  c->st_bin);
    k_st_class<<<nw, kBlock, 0, s>>>(v, inv(f.hbox), inv(f.vbox), inv(f.wbox), c->st_key, c->st_rb,
                                     c->st_rep, c->st_cnt);
    k_st_slots<<<1, kWave, 0, s>>>(c->st_cnt, c->st_slot, c->st_skey, c->st_maxslot, c->st_n);
    k_st_check<<<nw, kBlock, 0, s>>>(v, 1e-13 * f.radius, c->st_key, c->st_rb, c->st_rep, c->st_slot);
    unsigned char *plen = c->st_follow + N;
    k_st_follow<<<nt, 256, 0, s>>>(c->N, c->st_key, c->st_rb, c->st_follow, plen);
    k_st_cut<<<nt, 256, 0, s>>>(c->N, c->st_key, c->st_follow, plen);
    k_st_emit<true><<<nt, 256, 0, s>>>(v, bins, c->st_key, c->st_rb, c->st_rep, plen, c->st_bin,
                                       c->st_run, c->st_int, c->st_bnd, c->st_n);
    k_st_scan<<<1, 1024, 0, s>>>(nbin, c->st_bin, c->st_n);
    k_st_emit<false><<<nt, 256, 0, s>>>(v, bins, c->st_key, c->st_rb, c->st_rep, plen, c->st_bin,
                                        c->st_run, c->st_int, c->st_bnd, c->st_n);
    if (hipGetLastError() != hipSuccess) { c->err = "FP64 transport: classification failed"; return AB_ERR_HIP; }
    c->st_valid = true;
    return AB_OK;
}

int stencil_transport(ab_ctx *c, double dt, double tol, bool diag)
{
    if (!c->st_valid)
        if (int rc = stencil_prepare(c)) return rc;
    DevCloud v = c->view();
    hipStream_t s = c->stream;
    const ab_config &f = c->cfg;
    const int nchunk = (c->nodes + kWave - 1) / kWave;
    if (c->st_maxslot > 0)
    {
        k_stencil_coef<<<dim3(nchunk, c->st_maxslot), kWave, 0, s>>>(
            v, dt, f.radius, tol, f.mls_order, c->st_n, c->st_skey, c->st_rep, c->st_rb, nchunk,
            c->st_coef);
        const RunArgs a{c->g, c->gt, c->st_coef, c->st_rb, dt, f.radius, f.mls_clamp, c->mlsflag,
                        c->mlsovr};
        const long long items = (long long)c->N * nchunk;   // at most: one run per particle
        const int grid = (int)std::min<long long>((items + 31) / 32 * 8, 256 * 3);
        if (diag)
            k_apply_runs<true><<<grid, kBlock, 0, s>>>(v, a, c->st_n, c->st_run, c->st_key,
                                                       c->st_slot, nchunk);
        else
            k_apply_runs<false><<<grid, kBlock, 0, s>>>(v, a, c->st_n, c->st_run, c->st_key,
                                                        c->st_slot, nchunk);
    }
    launch_transport_fp64(v, c->g, c->gt, dt, f.radius, f.mls_order, tol, f.mls_clamp, c->mlsflag,
                          c->mlsovr, c->st_int, c->n_int, c->st_bnd, c->n_bnd, diag, s, nullptr,
                          c->st_n + N_INT);
    return hipGetLastError() == hipSuccess ? AB_OK : AB_ERR_HIP;
}

}  // namespace ab
