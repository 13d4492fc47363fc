// Dispersion: linear_dispersive_solver_mod.f90 without DISPERSIVE_PEREGRINE_IN_FLUX_FORM
// (the reference's default), staggered (leapfrog) and cell-centred (finite-volume) forms.
//
// solve_dispersive_terms (domain_mod.f90:4319-4343 -> linear_dispersive_solve_TRIDIAG,
// :1193-1354): the explicit part of the dispersive terms from the state stored before the
// shallow-water step and the right-hand side RHS = U - Ax (U itself on the border), the
// solution optionally extrapolated in time from three earlier levels
// (quadratic_extrapolation_mod.f90:91-193), then tridiagonal iterations: every row of UH
// (:663-790) and then every column of VH (:792-921) is one tridiagonal system, solved by
// LAPACK's dgtsv elimination with partial pivoting (the reference vendors it,
// util/lapack_tridiagonal_solves.f:462-673), a lane per row (UH) or column (VH).
#include <algorithm>

#include "swh_internal.h"

namespace swh {

namespace {

template <typename T>
__device__ __forceinline__ T dmax_d(T a, T b) { return a > b ? a : b; }
template <typename T>
__device__ __forceinline__ T dmin_d(T a, T b) { return a < b ? a : b; }

// depth at a UH / VH point: msl-relative, zero unless both cells are below msl (:209-210)
template <typename T>
__device__ __forceinline__ T disp_depth(T msl, T e1, T e2)
{
    return (e1 < msl && e2 < msl) ? T(0.5) * (msl - e1 + msl - e2) : T(0);
}

// cell-centred depth: msl-relative where the cell and its two neighbours along the line
// are all below msl (:451, :493)
template <typename T>
__device__ __forceinline__ T disp_depth_cc(T msl, T em, T e0, T ep)
{
    return (em < msl && e0 < msl && ep < msl) ? (msl - e0) : T(0);
}

template <typename T>
__device__ __forceinline__ T disp_premult(const DispArgs<T> &a, T dep, T r)
{
    return dep * dep / (T(3) * r) * dmin_d(T(1), dmax_d(T(0), (dep - a.td2) / (a.td1 - a.td2)));
}

// explicit part from the stored state (linear_dispersive_staggered_matmult, :182-417)
// and the right-hand side (:1226-1265), per cell
template <typename T>
__global__ void disp_rhs_kernel(DispArgs<T> a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i >= a.nx || j >= a.ny) return;
    const int nx = a.nx, ny = a.ny, P = a.pitch;
    const long long o = (long long)j * P + i;
    const bool edge = i == 0 || j == 0 || i == nx - 1 || j == ny - 1;
    if (edge) {
        a.RU[o] = a.UH[o];
        a.RV[o] = a.VH[o];
        return;
    }
    const T msl = a.msl, dlon = a.dlon, dlat = a.dlat, dle1 = (T)a.dle[0];
    const T *el = a.LE, *uh = a.LU, *vh = a.LV;
    if (a.cell) {
        // linear_dispersive_cellcentred_matmult (:419-660)
        const T dbe_jm = (T)a.dbe[j - 1], dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1], dbe_jpp = (T)a.dbe[j + 2];
        {
            const T Rdlon = T(0.5) * (dbe_jp + dbe_j);
            const T Rdlat = Rdlon * dlat / dlon;
            const T cjp1 = T(0.5) * (dbe_jpp + dbe_jp) * dlat / (dlon * dle1);
            const T cjm1 = T(0.5) * (dbe_j + dbe_jm) * dlat / (dlon * dle1);
            const T dep = disp_depth_cc(msl, el[o - 1], el[o], el[o + 1]);
            const T pm = disp_premult(a, dep, Rdlon);
            const T ax = pm * (T(1) / Rdlon * (uh[o + 1] - T(2) * uh[o] + uh[o - 1]) +
                               T(1) / Rdlat * ((cjp1 * vh[o + 1 + P] - cjm1 * vh[o + 1 - P]) * T(0.25) -
                                               (cjp1 * vh[o - 1 + P] - cjm1 * vh[o - 1 - P]) * T(0.25)));
            a.RU[o] = a.UH[o] - ax;
        }
        {
            const T r_dlat = dle1;
            const T Rdlon_jph = dbe_jp, Rdlon_jmh = dbe_j;
            const T Rdlat_jph = Rdlon_jph * dlat / dlon, Rdlat_jmh = Rdlon_jmh * dlat / dlon;
            const T cjp1 = T(0.5) * (dbe_jpp + dbe_jp) * dlat / (dle1 * dlon);
            const T cj = T(0.5) * (dbe_jp + dbe_j) * dlat / (dle1 * dlon);
            const T cjm1 = T(0.5) * (dbe_j + dbe_jm) * dlat / (dle1 * dlon);
            const T dep = disp_depth_cc(msl, el[o - P], el[o], el[o + P]);
            const T pm = disp_premult(a, dep, r_dlat);
            const T ax = pm * ((T(1) / Rdlon_jph * (uh[o + 1 + P] - uh[o - 1 + P] + uh[o + 1] - uh[o - 1]) * T(0.25) -
                                T(1) / Rdlon_jmh * (uh[o + 1 - P] - uh[o - 1 - P] + uh[o + 1] - uh[o - 1]) * T(0.25)) +
                               (T(1) / Rdlat_jph * (cjp1 * vh[o + P] - cj * vh[o]) -
                                T(1) / Rdlat_jmh * (cj * vh[o] - cjm1 * vh[o - P])));
            a.RV[o] = a.VH[o] - ax;
        }
        return;
    }
    // UH at (i+1/2, j)
    {
        const T dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1];
        const T Rdlon = T(0.5) * (dbe_jp + dbe_j);
        const T Rdlat = Rdlon * dlat / dlon;
        const T cjph = dbe_jp * dlat / (dlon * dle1);
        const T cjmh = dbe_j * dlat / (dlon * dle1);
        const T dep = disp_depth(msl, el[o], el[o + 1]);
        const T pm = disp_premult(a, dep, Rdlon);
        const T ax = pm * (T(1) / Rdlon * (uh[o + 1] - T(2) * uh[o] + uh[o - 1]) +
                           T(1) / Rdlat * ((cjph * vh[o + 1] - cjmh * vh[o + 1 - P]) - (cjph * vh[o] - cjmh * vh[o - P])));
        a.RU[o] = a.UH[o] - ax;
    }
    // VH at (i, j+1/2)
    {
        const T r_dlat = dle1;
        const T dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1], dbe_jpp = (T)a.dbe[j + 2];
        const T Rdlon_jp1 = T(0.5) * (dbe_jpp + dbe_jp);
        const T Rdlon_j = T(0.5) * (dbe_jp + dbe_j);
        const T Rdlat_jp1 = Rdlon_jp1 * dlat / dlon;
        const T Rdlat_j = Rdlon_j * dlat / dlon;
        const T cjp1h = dbe_jpp * dlat / (dle1 * dlon);
        const T cjph = dbe_jp * dlat / (dle1 * dlon);
        const T cjmh = dbe_j * dlat / (dle1 * dlon);
        const T dep = disp_depth(msl, el[o], el[o + P]);
        const T pm = disp_premult(a, dep, r_dlat);
        const T ax = pm * ((T(1) / Rdlon_jp1 * (uh[o + P] - uh[o + P - 1]) - T(1) / Rdlon_j * (uh[o] - uh[o - 1])) +
                           (T(1) / Rdlat_jp1 * (cjp1h * vh[o + P] - cjph * vh[o]) -
                            T(1) / Rdlat_j * (cjph * vh[o] - cjmh * vh[o - P])));
        a.RV[o] = a.VH[o] - ax;
    }
}

// quadratic extrapolation in time of UH and VH (all cells); the coefficients of
// extrapolate_in_time (quadratic_extrapolation_mod.f90:171-181) from the level times and
// the forward time, both on the device (finite-volume times never leave it)
template <typename T>
__global__ void disp_extrapolate_kernel(DispArgs<T> a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i >= a.nx || j >= a.ny) return;
    const double t_fwd = a.sc ? a.sc->time : a.t_fwd;
    const double tn2 = a.qt[0] - a.qt[2], tn1 = a.qt[1] - a.qt[2], t1 = t_fwd - a.qt[2];
    const double pm = 1.0 / (tn1 * (tn2 * tn2) - tn2 * (tn1 * tn1));
    const T ca = (T)(1.0 + t1 * pm * (-(tn2 * tn2) + tn1 * tn1) + (t1 * t1) * pm * (tn2 - tn1));
    const T cb = (T)(t1 * pm * (tn2 * tn2) + (t1 * t1) * pm * (-tn2));
    const T cc = (T)(t1 * pm * (-(tn1 * tn1)) + (t1 * t1) * pm * tn1);
    const long long o = (long long)j * a.pitch + i, P2 = (long long)a.pitch * a.ny;
    a.UH[o] = a.Y0[o] * ca + a.Y1[o] * cb + a.Y2[o] * cc;
    a.VH[o] = a.Y0[o + P2] * ca + a.Y1[o + P2] * cb + a.Y2[o + P2] * cc;
}

// ---- the tridiagonal solves -----------------------------------------------------------
//
// dgtsv's elimination splits into a part that the matrix alone decides (the multipliers,
// the row swaps, the eliminated coefficients), done once per solve, and the part that
// carries the right-hand side, done in every iteration; each keeps dgtsv's operations
// and their order, so the results are its bits. Work is laid out element-major: element
// k of line l at (k * lines + l), lines being the rows j of UH or the columns i of VH,
// so a wavefront's 64 lines touch neighbouring addresses at every element of the walk.
//
// What bounds it: a walk is serial along its line and there are only as many lanes as
// lines (11 wavefronts on a 700 x 517 grid), so its time is the chain of dependent
// operations per element. Everything that is not part of that chain is out of it:
// coefficients and right-hand sides are formed by kernels with a thread per cell (the UH
// ones transposed through LDS), coefficients are packed so that an element is one or two
// wide loads, which wavefronts of their own bring into LDS ahead of the computing one
// (walk_phases), and the division of the back substitution is by a reciprocal formed
// beforehand (div_by). 700 x 517 FP64: a walk takes 46 us (53 with 64 lines to a workgroup
// instead of 16), the elimination of both directions 92 us once per solve, where a sweep with
// a lane doing all of a line's work took 1170 and 1360 us; a dispersive step (two iterations)
// 480 us, 5.2 ms before. The matrices take six values per
// element and direction: 13 planes of work with the right-hand side, where the sweeps needed
// 4. Where those don't fit in device memory, the directions share a place (7 planes) and every
// iteration eliminates anew: the same bits, a step of 0.65 ms takes 1.09.
constexpr int kTile = 32;    // tile of the transposing kernels

template <typename T>
struct Coef4 {   // raw: {diagonal, below, above, -}; eliminated: {diagonal, 1 / diagonal, above, second above}
    T x, y, z, w;
};
template <typename T>
struct Coef2 {   // {multiplier of the elimination step, 1 if it swapped rows}
    T x, y;
};

template <typename T>
struct DispWork {
    Coef4<T> *c4[2];   // UH lines, VH lines
    Coef2<T> *c2[2];
    T *b;              // right-hand side and solution of the sweep at hand
};

template <typename T>
__host__ __device__ inline DispWork<T> disp_work(const DispArgs<T> &a)
{
    const long long n = (long long)a.nx * a.ny;
    DispWork<T> w;
    w.c4[0] = (Coef4<T> *)a.W;
    w.c4[1] = w.c4[0] + a.second;
    w.c2[0] = (Coef2<T> *)(w.c4[1] + n);
    w.c2[1] = w.c2[0] + a.second;
    w.b = (T *)(w.c2[1] + n);
    return w;
}

__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// x / d from r = 1 / d rounded to nearest: one refinement makes the quotient faithful, the
// second rounds it correctly (Markstein, IBM J. Res. Dev. 34, 1990), so it is the bits of
// x / d where no intermediate leaves the normal range (disp_walk_kernel checks that). Five
// dependent operations instead of the division's twelve or so.
template <typename T>
__device__ __forceinline__ T div_by(T x, T d, T r)
{
    T q = x * r;
    q = fma_t(fma_t(-d, q, x), r, q);
    return fma_t(fma_t(-d, q, x), r, q);
}

// coefficients of UH's row j at cell i (:663-790; cell-centred :961-997)
template <typename T>
__device__ __forceinline__ Coef4<T> uh_coef(const DispArgs<T> &a, int i, int j)
{
    if (i == 0 || i == a.nx - 1) return Coef4<T>{T(1), T(0), T(0), T(0)};
    const T dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1];
    const T Rdlon = T(0.5) * (dbe_jp + dbe_j);
    const long long o = (long long)j * a.pitch + i;
    const T dep = a.cell ? disp_depth_cc(a.msl, a.E[o - 1], a.E[o], a.E[o + 1]) : disp_depth(a.msl, a.E[o], a.E[o + 1]);
    const T pm = disp_premult(a, dep, Rdlon);
    return Coef4<T>{T(1) + T(2) * pm * T(1) / Rdlon, -pm * T(1) / Rdlon, -pm * T(1) / Rdlon, T(0)};
}

// the right-hand side there, from the current VH
template <typename T>
__device__ __forceinline__ T uh_rhs(const DispArgs<T> &a, int i, int j)
{
    const int P = a.pitch;
    const long long o = (long long)j * P + i;
    if (i == 0 || i == a.nx - 1) return a.RU[o];
    const T msl = a.msl, dlon = a.dlon, dlat = a.dlat, dle1 = (T)a.dle[0];
    const T dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1];
    const T Rdlon = T(0.5) * (dbe_jp + dbe_j);
    const T Rdlat = Rdlon * dlat / dlon;
    if (a.cell) {
        const T cjp1 = T(0.5) * ((T)a.dbe[j + 2] + dbe_jp) * dlat / (dlon * dle1);
        const T cjm1 = T(0.5) * (dbe_j + (T)a.dbe[j - 1]) * dlat / (dlon * dle1);
        const T pm = disp_premult(a, disp_depth_cc(msl, a.E[o - 1], a.E[o], a.E[o + 1]), Rdlon);
        return a.RU[o] + pm * (T(1) / Rdlat * ((cjp1 * a.VH[o + 1 + P] - cjm1 * a.VH[o + 1 - P]) * T(0.25) -
                                               (cjp1 * a.VH[o - 1 + P] - cjm1 * a.VH[o - 1 - P]) * T(0.25)));
    }
    const T cjph = dbe_jp * dlat / (dlon * dle1);
    const T cjmh = dbe_j * dlat / (dlon * dle1);
    const T pm = disp_premult(a, disp_depth(msl, a.E[o], a.E[o + 1]), Rdlon);
    return a.RU[o] + pm * (T(1) / Rdlat * ((cjph * a.VH[o + 1] - cjmh * a.VH[o + 1 - P]) -
                                           (cjph * a.VH[o] - cjmh * a.VH[o - P])));
}

// coefficients of VH's column i at cell j (:792-921; cell-centred :1101-1180)
template <typename T>
__device__ __forceinline__ Coef4<T> vh_coef(const DispArgs<T> &a, int i, int j)
{
    if (j == 0 || j == a.ny - 1) return Coef4<T>{T(1), T(0), T(0), T(0)};
    const int P = a.pitch;
    const long long o = (long long)j * P + i;
    const T msl = a.msl, dlon = a.dlon, dlat = a.dlat, dle1 = (T)a.dle[0];
    const T r_dlat = dle1;
    const T dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1], dbe_jpp = (T)a.dbe[j + 2];
    Coef4<T> c;
    c.w = T(0);
    if (a.cell) {
        const T Rdlat_jph = dbe_jp * dlat / dlon, Rdlat_jmh = dbe_j * dlat / dlon;
        const T cjp1 = T(0.5) * (dbe_jpp + dbe_jp) * dlat / (dle1 * dlon);
        const T cj = T(0.5) * (dbe_jp + dbe_j) * dlat / (dle1 * dlon);
        const T cjm1 = T(0.5) * (dbe_j + (T)a.dbe[j - 1]) * dlat / (dle1 * dlon);
        const T pm = disp_premult(a, disp_depth_cc(msl, a.E[o - P], a.E[o], a.E[o + P]), r_dlat);
        c.x = T(1) + pm * (T(1) / Rdlat_jph * cj + T(1) / Rdlat_jmh * cj);
        c.y = -pm * T(1) / Rdlat_jmh * cjm1;
        c.z = -pm * T(1) / Rdlat_jph * cjp1;
        return c;
    }
    const T Rdlat_jp1 = T(0.5) * (dbe_jpp + dbe_jp) * dlat / dlon;
    const T Rdlat_j = T(0.5) * (dbe_jp + dbe_j) * dlat / dlon;
    const T cjp1h = dbe_jpp * dlat / (dle1 * dlon);
    const T cjph = dbe_jp * dlat / (dle1 * dlon);
    const T cjmh = dbe_j * dlat / (dle1 * dlon);
    const T pm = disp_premult(a, disp_depth(msl, a.E[o], a.E[o + P]), r_dlat);
    c.x = T(1) + pm * (T(1) / Rdlat_jp1 * cjph + T(1) / Rdlat_j * cjph);
    c.y = -pm * T(1) / Rdlat_j * cjmh;
    c.z = -pm * T(1) / Rdlat_jp1 * cjp1h;
    return c;
}

template <typename T>
__device__ __forceinline__ T vh_rhs(const DispArgs<T> &a, int i, int j)
{
    const int P = a.pitch;
    const long long o = (long long)j * P + i;
    if (j == 0 || j == a.ny - 1) return a.RV[o];
    const T r_dlat = (T)a.dle[0];
    const T dbe_j = (T)a.dbe[j], dbe_jp = (T)a.dbe[j + 1];
    if (a.cell) {
        const T pm = disp_premult(a, disp_depth_cc(a.msl, a.E[o - P], a.E[o], a.E[o + P]), r_dlat);
        return a.RV[o] + pm * ((T(1) / dbe_jp *
                                    (a.UH[o + 1 + P] - a.UH[o - 1 + P] + a.UH[o + 1] - a.UH[o - 1]) * T(0.25) -
                                T(1) / dbe_j *
                                    (a.UH[o + 1 - P] - a.UH[o - 1 - P] + a.UH[o + 1] - a.UH[o - 1]) * T(0.25)));
    }
    const T Rdlon_jp1 = T(0.5) * ((T)a.dbe[j + 2] + dbe_jp);
    const T Rdlon_j = T(0.5) * (dbe_jp + dbe_j);
    const T pm = disp_premult(a, disp_depth(a.msl, a.E[o], a.E[o + P]), r_dlat);
    return a.RV[o] + pm * ((T(1) / Rdlon_jp1 * (a.UH[o + P] - a.UH[o + P - 1]) -
                            T(1) / Rdlon_j * (a.UH[o] - a.UH[o - 1])));
}

// The matrices, a thread per cell, of direction dir0 + blockIdx.z: 0 the rows of UH
// (j = 1 .. ny-2, transposed to element i, line j through LDS), 1 the columns of VH.
template <typename T>
__global__ __launch_bounds__(256) void disp_coef_kernel(DispArgs<T> a, int dir0)
{
    const DispWork<T> w = disp_work(a);
    const int i0 = blockIdx.x * kTile, j0 = blockIdx.y * kTile;
    const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;
    if (dir0 + (int)blockIdx.z == 1) {
        const int i = i0 + tx;
        for (int r = ty; r < kTile; r += 256 / kTile) {
            const int j = j0 + r;
            if (i >= 1 && i <= a.nx - 2 && j < a.ny) {
                w.c4[1][(long long)j * a.nx + i] = vh_coef(a, i, j);
                w.c2[1][(long long)j * a.nx + i] = Coef2<T>{T(0), T(0)};
            }
        }
        return;
    }
    __shared__ Coef4<T> tile[kTile][kTile + 1];
    for (int r = ty; r < kTile; r += 256 / kTile) {
        const int i = i0 + tx, j = j0 + r;
        if (i < a.nx && j >= 1 && j <= a.ny - 2) tile[r][tx] = uh_coef(a, i, j);
    }
    __syncthreads();
    for (int r = ty; r < kTile; r += 256 / kTile) {
        const int i = i0 + r, j = j0 + tx;
        if (i < a.nx && j >= 1 && j <= a.ny - 2) {
            w.c4[0][(long long)i * a.ny + j] = tile[tx][r];
            w.c2[0][(long long)i * a.ny + j] = Coef2<T>{T(0), T(0)};
        }
    }
}

// A workgroup walks kLines lines, a lane per line of wavefront 0, which computes; the other
// wavefronts load. The walk goes in phases of C elements; a pair of loader wavefronts takes
// every kPairs'th phase, half its elements each: it holds them in registers while they
// travel (kPairs - 1 phases long), puts them into one of two LDS buffers in the phase before
// their use, and starts its next ones after the barrier, where nobody waits for their
// issue. The computing wavefront thus reads only LDS, and its chain of dependent
// operations never waits for memory (written by other XCDs: near a microsecond): 46 us for
// a walk of 600 elements, against 87 us with the same wavefront's loads two chunks ahead in
// registers and 145 us one chunk ahead. 16 lines to a workgroup, not 64: four times as many
// CUs work (46 against 53 us).
constexpr int kLines = 16;
constexpr int kPairs = 3;
constexpr int kWalkThreads = 64 * (2 * kPairs + 1);

// p[line] by a 32-bit byte offset: the row's address stays in scalar registers (no 64-bit
// vector additions in the computing wavefront)
template <typename T>
__device__ __forceinline__ T &at(T *p, unsigned off) { return *(T *)((char *)p + off); }

// Workgroup barrier that orders LDS only: the loaders' loads stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 'phases' phases: load(phase, half) brings half a phase's elements into the loader's
// registers, put(half, buffer) stores them to LDS, use(phase, buffer) computes with them.
template <typename Load, typename Put, typename Use>
__device__ __forceinline__ void walk_phases(int phases, Load load, Put put, Use use)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // (uniform: scalar branches)
    if (wave > 0) {
        const int half = (wave - 1) & 1;
        int mine = (wave - 1) >> 1;   // the phase in this loader's registers
        if (mine < phases) load(mine, half);
        for (int p = -1; p < phases; p++) {
            // between two barriers: phase p is computed, phase p + 1 put into LDS
            const bool turn = mine == p + 1 && mine < phases;
            if (turn) put(half, mine & 1);
            lds_barrier();
            if (turn) {
                mine += kPairs;
                if (mine < phases) load(mine, half);
            }
        }
    } else {
        lds_barrier();
        for (int p = 0; p < phases; p++) {
            use(p, p & 1);
            lds_barrier();
        }
    }
}

// The elimination of the matrices: the first workgroups the rows of UH, the others the
// columns of VH. dgtsv's two branches per element; where it would stop at a zero pivot, no
// further step changes anything and the line is not substituted back (its last reciprocal
// is -inf). A lone computing wavefront is bound by the instructions it issues (4 cycles
// each) as much as by its chain, so the swap-free step, which is nearly every one, is
// its own branch.
template <typename T>
__global__ __launch_bounds__(kWalkThreads) void disp_factor_kernel(DispArgs<T> a, int blocks_uh)
{
    constexpr int C = 8;
    __shared__ T buf[2][C][3][kLines];
    const DispWork<T> w = disp_work(a);
    const int dir = (int)blockIdx.x >= blocks_uh ? 1 : 0, lane = threadIdx.x % kLines;
    const int sub = (threadIdx.x & 63) / kLines;   // which of the elements that a loader takes at once
    const int n = dir ? a.ny : a.nx, lines = dir ? a.nx : a.ny;
    // (lanes past the last line repeat it: the same values to the same places)
    const unsigned line = min(1 + ((int)blockIdx.x - (dir ? blocks_uh : 0)) * kLines + lane, lines - 2);
    const long long s = lines;
    Coef4<T> *const c4 = w.c4[dir];
    Coef2<T> *const c2 = w.c2[dir];
    const unsigned off4 = line * (unsigned)sizeof(Coef4<T>);
    T dg = c4[line].x, du = c4[line].z;
    bool stop = false;
    int after_swap = 0;   // the step before changed this one's superdiagonal
    constexpr int CH = C / 2, CL = CH * kLines / 64;   // elements per half phase, per loader lane
    T r[CL][3];
    // element k + 1 of the raw matrix enters at step k (ahead of what is written)
    walk_phases(
        (n - 1 + C - 1) / C,
        [&](int p, int half) {
#pragma unroll
            for (int u = 0; u < CL; u++) {
                const Coef4<T> q = c4[(long long)min(p * C + half * CH + u * (64 / kLines) + sub + 1, n - 1) * s + line];
                r[u][0] = q.x; r[u][1] = q.y; r[u][2] = q.z;
            }
        },
        [&](int half, int b) {
#pragma unroll
            for (int u = 0; u < CL; u++)
#pragma unroll
                for (int v = 0; v < 3; v++) buf[b][half * CH + u * (64 / kLines) + sub][v][lane] = r[u][v];
        },
        [&](int p, int b) {
            Coef4<T> *o4 = c4 + (long long)p * C * s;
            Coef2<T> *o2 = c2 + (long long)p * C * s;
            T in[C][3];
#pragma unroll
            for (int u = 0; u < C; u++)
#pragma unroll
                for (int v = 0; v < 3; v++) in[u][v] = buf[b][u][v][lane];
#pragma unroll
            for (int u = 0; u < C; u++) {
                const T dg1 = in[u][0], dl = in[u][1], du1 = in[u][2];
                if (p * C + u >= n - 1) break;
                bool sw = !(fabs(dg) >= fabs(dl));
                if (__builtin_expect(__any(sw | stop | (dg == T(0))) | after_swap, 0)) {
                    after_swap = __any(sw);
                    sw = sw && !stop;
                    stop = stop || (!sw && dg == T(0));
                    Coef4<T> q{dg, T(0), du, T(0)};
                    Coef2<T> f{T(0), T(0)};
                    f.x = stop ? T(0) : (sw ? dg : dl) / (sw ? dl : dg);
                    const bool second = sw && p * C + u < n - 2;
                    if (sw) { q.x = dl; q.z = dg1; f.y = T(1); }
                    if (second) q.w = du1;
                    dg = (sw ? du : dg1) - f.x * (sw ? dg1 : du);
                    du = second ? -f.x * du1 : du1;
                    o4[line] = q;
                    o2[line] = f;
                } else {
                    // (the superdiagonal, its zero neighbour and the swap flag stand)
                    const T fact = dl / dg;
                    at(o4, off4).x = dg;
                    at(o2, off4 / 2).x = fact;
                    dg = dg1 - fact * du;
                    du = du1;
                }
                o4 += s;
                o2 += s;
            }
        });
    if (threadIdx.x < kLines)
        (c4 + (long long)(n - 1) * s)[line] =
            Coef4<T>{dg, (stop || dg == T(0)) ? -T(__builtin_huge_val()) : T(0), T(0), T(0)};
}

// the reciprocals of the eliminated diagonals (NaN where div_by does not hold), a thread
// per cell: off the elimination's chain
template <typename T>
__global__ __launch_bounds__(256) void disp_recip_kernel(DispArgs<T> a, int dir0)
{
    const DispWork<T> w = disp_work(a);
    const int dir = dir0 + (int)blockIdx.z, n = dir ? a.ny : a.nx, lines = dir ? a.nx : a.ny;
    const int line = 1 + blockIdx.x * 256 + threadIdx.x, k = blockIdx.y;
    if (line > lines - 2 || k >= n - 1) return;
    Coef4<T> *q = w.c4[dir] + (long long)k * lines + line;
    const T d = q->x, ad = fabs(d), lim = sizeof(T) == 8 ? T(0x1p100) : T(0x1p20f);
    q->y = (ad < lim && ad * lim > T(1)) ? T(1) / d : T(__builtin_nan(""));
}

// right-hand sides of UH's rows, transposed as the matrix
template <typename T>
__global__ __launch_bounds__(256) void disp_uh_rhs_kernel(DispArgs<T> a)
{
    __shared__ T tile[kTile][kTile + 1];
    T *b = disp_work(a).b;
    const int i0 = blockIdx.x * kTile, j0 = blockIdx.y * kTile;
    const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;
    for (int r = ty; r < kTile; r += 256 / kTile) {
        const int i = i0 + tx, j = j0 + r;
        if (i < a.nx && j >= 1 && j <= a.ny - 2) tile[r][tx] = uh_rhs(a, i, j);
    }
    __syncthreads();
    for (int r = ty; r < kTile; r += 256 / kTile) {
        const int i = i0 + r, j = j0 + tx;
        if (i < a.nx && j >= 1 && j <= a.ny - 2) b[(long long)i * a.ny + j] = tile[tx][r];
    }
}

// the solved rows of UH back from the transposed work array
template <typename T>
__global__ __launch_bounds__(256) void disp_uh_put_kernel(DispArgs<T> a)
{
    __shared__ T tile[kTile][kTile + 1];
    const T *b = disp_work(a).b;
    const int i0 = blockIdx.x * kTile, j0 = blockIdx.y * kTile;
    const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;
    for (int r = ty; r < kTile; r += 256 / kTile) {
        const int i = i0 + r, j = j0 + tx;
        if (i < a.nx && j >= 1 && j <= a.ny - 2) tile[tx][r] = b[(long long)i * a.ny + j];
    }
    __syncthreads();
    for (int r = ty; r < kTile; r += 256 / kTile) {
        const int i = i0 + tx, j = j0 + r;
        if (i < a.nx && j >= 1 && j <= a.ny - 2) a.UH[(long long)j * a.pitch + i] = tile[r][tx];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void disp_vh_rhs_kernel(DispArgs<T> a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i < 1 || i > a.nx - 2) return;
    disp_work(a).b[(long long)j * a.nx + i] = vh_rhs(a, i, j);
}

__device__ __forceinline__ int exponent_of(double x) { return __builtin_amdgcn_frexp_exp(x); }
__device__ __forceinline__ int exponent_of(float x) { return __builtin_amdgcn_frexp_expf(x); }

// The right-hand side through the elimination and the back substitution (b: work element
// k of line l at k * lines + l); the solution goes to out + k * so. The loaders tell the
// computing wavefront which phases hold a row swap, so that the others run without its
// selections and without the second superdiagonal (0 there: subtracting 0 * x changes
// nothing for finite x, and phases with other values run again in full).
template <typename T>
__global__ __launch_bounds__(kWalkThreads) void disp_walk_kernel(const Coef4<T> *__restrict__ c4,
                                                                 const Coef2<T> *__restrict__ c2, T *b, int n,
                                                                 int lines, T *out, long long so)
{
    constexpr int C = 64, B = 16;   // elements per phase, per unrolled block
    __shared__ Coef2<T> cbuf[2][C][2][kLines];
    __shared__ T bbuf[2][C][kLines];
    __shared__ int swaps[2][2];
    const int lane = threadIdx.x % kLines;
    const int sub = (threadIdx.x & 63) / kLines;   // which of the elements that a loader takes at once
    // (lanes past the last line repeat it: the same values to the same places)
    const unsigned line = min(1 + (int)blockIdx.x * kLines + lane, lines - 2);
    const long long s = lines;
    const unsigned off = line * (unsigned)sizeof(T);
    T bc = b[line];
    constexpr int CH = C / 2, CL = CH * kLines / 64;   // elements per half phase, per loader lane
    Coef2<T> r[CL][2];
    T rb[CL];
    // step k: b(k + 1) -= multiplier * b(k), with the rows swapped where the matrix's
    // elimination swapped them; b(k) is final after it (the elements being loaded are ahead
    // of the ones written)
    walk_phases(
        (n - 1 + C - 1) / C,
        [&](int p, int half) {
#pragma unroll
            for (int u = 0; u < CL; u++) {
                const long long k = min(p * C + half * CH + u * (64 / kLines) + sub, n - 2);
                r[u][0] = c2[k * s + line];
                rb[u] = b[(k + 1) * s + line];
            }
        },
        [&](int half, int q) {
            bool any = false;
#pragma unroll
            for (int u = 0; u < CL; u++) {
                const int e = half * CH + u * (64 / kLines) + sub;
                cbuf[q][e][0][lane] = r[u][0];
                bbuf[q][e][lane] = rb[u];
                any = any | (r[u][0].y != T(0));
            }
            const int sw = __any(any);
            if ((threadIdx.x & 63) == 0) swaps[q][half] = sw;
        },
        [&](int p, int q) {
            T *bo = b + (long long)p * C * s;
            const bool swap_free = !__builtin_amdgcn_readfirstlane(swaps[q][0] | swaps[q][1]);
            const int m = min(C, n - 1 - p * C);
            auto block = [&](int u0) {
                T f[B], x[B];
#pragma unroll
                for (int u = 0; u < B; u++) { f[u] = cbuf[q][u0 + u][0][lane].x; x[u] = bbuf[q][u0 + u][lane]; }
#pragma unroll
                for (int u = 0; u < B; u++) {
                    at(bo, off) = bc;
                    bo += s;
                    bc = x[u] - f[u] * bc;
                }
            };
            int u = 0;
            if (swap_free && m == C) {
#pragma unroll
                for (; u < C; u += B) block(u);
            } else if (swap_free) {
                for (; u + B <= m; u += B) block(u);
            }
            for (; u < m; u++) {
                const Coef2<T> f = cbuf[q][u][0][lane];
                const T x = bbuf[q][u][lane];
                const bool sw = f.y != T(0);
                const T bk = sw ? x : bc, rest = sw ? bc : x;
                at(bo, off) = bk;
                bo += s;
                bc = rest - f.x * bk;
            }
        });
    // dgtsv stopped at a zero pivot: the eliminated right-hand side stands as it is
    const Coef4<T> last = (c4 + (long long)(n - 1) * s)[line];
    const bool dead = last.y == -T(__builtin_huge_val());
    const int any_dead = __any(dead);
    // (x(n-2) has no second superdiagonal: its coefficient is 0)
    T x1 = dead ? bc : bc / last.x, x2 = T(0);
    if (threadIdx.x < kLines) (out + (long long)(n - 1) * so)[line] = x1;
    __syncthreads();   // the loaders read what was written above
    walk_phases(
        (n - 1 + C - 1) / C,   // elements n - 2, n - 3, ..., 0
        [&](int p, int half) {
#pragma unroll
            for (int u = 0; u < CL; u++) {
                const long long k = max(n - 2 - (p * C + half * CH + u * (64 / kLines) + sub), 0);
                const Coef4<T> q = c4[k * s + line];
                r[u][0] = Coef2<T>{q.x, q.y};
                r[u][1] = Coef2<T>{q.z, q.w};
                rb[u] = b[k * s + line];
            }
        },
        [&](int half, int q) {
            bool any = false;
#pragma unroll
            for (int u = 0; u < CL; u++) {
                const int e = half * CH + u * (64 / kLines) + sub;
                cbuf[q][e][0][lane] = r[u][0];
                cbuf[q][e][1][lane] = r[u][1];
                bbuf[q][e][lane] = rb[u];
                any = any | (r[u][1].y != T(0));
            }
            const int sw = __any(any);
            if ((threadIdx.x & 63) == 0) swaps[q][half] = sw;
        },
        [&](int p, int q) {
            T *const o0 = out + (long long)(n - 2 - p * C) * so;
            T *oo = o0;
            const T x1s = x1, x2s = x2;
            const bool swap_free = !any_dead && !__builtin_amdgcn_readfirstlane(swaps[q][0] | swaps[q][1]);
            const int m = min(C, n - 1 - p * C);
            int lo = 0;
            auto block = [&](int u0) {
                Coef2<T> d[B];
                T up[B], v[B];
#pragma unroll
                for (int u = 0; u < B; u++) {
                    d[u] = cbuf[q][u0 + u][0][lane];
                    up[u] = cbuf[q][u0 + u][1][lane].x;
                    v[u] = bbuf[q][u0 + u][lane];
                }
#pragma unroll
                for (int u = 0; u < B; u++) {
                    const T t = v[u] - up[u] * x1;
                    lo = min(lo, exponent_of(t));   // (0 for t == 0)
                    x2 = x1;
                    x1 = div_by(t, d[u].x, d[u].y);
                    at(oo, off) = x1;
                    oo -= so;
                }
            };
            int u = 0;
            if (swap_free && m == C) {
#pragma unroll
                for (; u < C; u += B) block(u);
            } else if (swap_free) {
                for (; u + B <= m; u += B) block(u);
            }
            // div_by holds unless a numerator is tiny; where one or a divisor is huge, not
            // finite or out of range, a NaN has come through to x1
            if (u && __any(lo < (sizeof(T) == 8 ? -900 : -90) || !(x1 == x1))) {
                x1 = x1s; x2 = x2s;
                oo = o0;
                u = 0;
            }
            for (; u < m; u++) {
                const Coef2<T> d = cbuf[q][u][0][lane], e = cbuf[q][u][1][lane];
                const T v = bbuf[q][u][lane];
                const T y = (v - e.x * x1 - e.y * x2) / d.x;
                at(oo, off) = dead ? v : y;
                oo -= so;
                x2 = x1;
                x1 = y;
            }
        });
}

}  // namespace

__global__ void disp_qt_append_kernel(double *qt, const DevScalars *sc, double t_host)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    qt[0] = qt[1];
    qt[1] = qt[2];
    qt[2] = sc ? sc->time : t_host;
}

template <typename T>
hipError_t launch_dispersion(const DispArgs<T> &a, int make_rhs, int extrapolate, int niter, hipStream_t s)
{
    if (a.nx < 3 || a.ny < 3) return hipErrorInvalidValue;
    const dim3 grid((a.nx + 255) / 256, a.ny), block(256);
    if (make_rhs) hipLaunchKernelGGL(disp_rhs_kernel<T>, grid, block, 0, s, a);
    if (extrapolate) hipLaunchKernelGGL(disp_extrapolate_kernel<T>, grid, block, 0, s, a);
    const dim3 tiles((a.nx + kTile - 1) / kTile, (a.ny + kTile - 1) / kTile);
    const int bu = (a.ny - 2 + kLines - 1) / kLines, bv = (a.nx - 2 + kLines - 1) / kLines;
    const DispWork<T> w = disp_work(a);
    // the matrices of 'dirs' directions from dir0, eliminated
    const auto matrices = [&](int dir0, int dirs) {
        const int rows = dir0 ? 0 : bu, columns = dir0 + dirs > 1 ? bv : 0, most = std::max(a.nx, a.ny);
        hipLaunchKernelGGL(disp_coef_kernel<T>, dim3(tiles.x, tiles.y, dirs), block, 0, s, a, dir0);
        hipLaunchKernelGGL(disp_factor_kernel<T>, dim3(rows + columns), dim3(kWalkThreads), 0, s, a, rows);
        hipLaunchKernelGGL(disp_recip_kernel<T>, dim3((most + 255) / 256, most, dirs), block, 0, s, a, dir0);
    };
    // (the elevation may have changed since the last solve)
    if (niter > 0 && a.second) matrices(0, 2);
    for (int it = 0; it < niter; it++) {
        if (!a.second) matrices(0, 1);
        hipLaunchKernelGGL(disp_uh_rhs_kernel<T>, tiles, block, 0, s, a);
        hipLaunchKernelGGL(disp_walk_kernel<T>, dim3(bu), dim3(kWalkThreads), 0, s, (const Coef4<T> *)w.c4[0],
                           (const Coef2<T> *)w.c2[0], w.b, a.nx, a.ny, w.b, (long long)a.ny);
        hipLaunchKernelGGL(disp_uh_put_kernel<T>, tiles, block, 0, s, a);
        if (!a.second) matrices(1, 1);
        hipLaunchKernelGGL(disp_vh_rhs_kernel<T>, grid, block, 0, s, a);
        hipLaunchKernelGGL(disp_walk_kernel<T>, dim3(bv), dim3(kWalkThreads), 0, s, (const Coef4<T> *)w.c4[1],
                           (const Coef2<T> *)w.c2[1], w.b, a.ny, a.nx, a.VH, (long long)a.pitch);
    }
    return hipGetLastError();
}

size_t dispersion_work_elems(int nx, int ny, bool compact) { return (compact ? 7 : 13) * (size_t)nx * ny; }

template hipError_t launch_dispersion<double>(const DispArgs<double> &, int, int, int, hipStream_t);
template hipError_t launch_dispersion<float>(const DispArgs<float> &, int, int, int, hipStream_t);

hipError_t launch_dispersion_qt_append(double *qt, const DevScalars *sc, double t_host, hipStream_t s)
{
    hipLaunchKernelGGL(disp_qt_append_kernel, dim3(1), dim3(64), 0, s, qt, sc, t_host);
    return hipGetLastError();
}

}  // namespace swh
