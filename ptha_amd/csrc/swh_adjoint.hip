// Discrete adjoint (exact transpose) of the truely-linear leapfrog step.
//
// The forward step (domain_mod_linear_solver_include.f90:92-113, 211-571 with
// truely_linear, Coriolis and linear drag, walls / no stage boundary) is linear in
// x = (S, UH, VH):  S' = S + D(UH, VH) on interior cells;
//   UH' = LF * (UH - aU (S'(i+1) - S'(i)) + bU * [VH(i,jm) + VH(i+1,jm) + VH(i,j) + VH(i+1,j)])
//   VH' = LF * (VH - aV (S'(j+1) - S'(j)) - bV * [UH(i,j) + UH(im,j) + UH(i,j+1) + UH(im,j+1)])
// on 0 <= i < nx-1, 0 <= j < ny-1 (jm = max(j-1,0), im = max(i-1,0)), identity
// elsewhere, with aU = cu(j) h_iph dle(i+1), aV = cv(j) h_jph dbe(j+1),
// bU = fu(j) [h_iph > 0] / 2, bV = fv(j) [h_jph > 0] / 2, LF = 1/(1 + dt*lfc).
// Given the adjoints (lS', lU', lV') of the outputs, the adjoints of the inputs are
//   pass 1:  lS  = lS' + sum over momentum points of the pressure-gradient transpose
//   pass 2:  lU, lV = identity/Coriolis transpose of (mu = LF*l') + divergence
//            transpose of lS,
// each a gather over +-1 neighbours, so no atomics are needed.

#include "swh_internal.h"
#include "swh_lanes.h"
#include "swh_launch.h"

namespace swh {

namespace {

constexpr int kAdjOwn = 61;   // columns a wavefront writes (lanes 1..61)

// Lane shifts across the wavefront; every lane must execute them.
template <typename T>
__device__ __forceinline__ T shl1(T v) { return lane_east(v); }   // value of lane + 1
template <typename T>
__device__ __forceinline__ T shr1(T v) { return lane_west(v); }   // value of lane - 1

// h_iph / h_jph of the truely-linear scheme (include.f90:265-280) from the elevations of
// the two cells of the face (e_far the east or north one)
template <typename T>
__device__ __forceinline__ T face_depth(T e0, T e_far, T msl)
{
    const T MIN = T(kMinDepth);
    return (e0 < -MIN + msl && e_far < -MIN + msl) ? msl - T(0.5) * (e_far + e0) : T(0);
}

}  // namespace

// One transposed step, fused and column-marching. Each lane owns one column (a
// wavefront owns 61: lane 0 is the western halo, lanes 62-63 the eastern one) and
// marches up a strip of rows, keeping what two rows share in registers; east and west
// neighbours come from the adjacent lanes. At row m (loaded now) it forms
//   h_iph(m), aU mu_U(m) = cu h_iph dle(i+1) LF lU,      (and its west neighbour's)
//   h_jph(m-1), aV mu_V(m-1) = cv h_jph dbe(j+1) LF lV,
//   the Coriolis products bU mu_U(m), bV mu_V(m-1) and their west / east neighbours',
//   pass 1 at row m-1: lS_in = lS + aU mu_U(i) - aU mu_U(i-1) + aV mu_V(j) - aV mu_V(j-1),
//   pass 2 at row m-2: lU_in, lV_in = identity / Coriolis transpose of LF l' plus the
//   divergence transpose of lS_in (its own, its east neighbour's, the row above's),
// with the operations and their order of the two-pass form, on 0 <= i < nx-1,
// 0 <= j < ny-1 for the momentum points and the interior for the stage: a term of a point
// outside is zeroed where it is formed. Each strip recomputes one row below and two above it.
//
// What bounds it: on grids of up to about 1024 x 1024 the chain of one strip's rows, so a row
// is short: each product is formed once, by the lane and in the row that it belongs to (its
// neighbour's is a lane move, the other row's is carried), 75 vector operations in FP32
// (85 at the grid's edges) against 163 when every term was formed where it is used; and the
// loads of the next two rows are issued before two rows are computed and looked at after
// them. 1024 x 1024 FP32 13.0 -> 8.9 us a step, 300 x 300 6.1 -> 4.3.
// Row coefficients of row r (loaded once per row at a clamped index, carried while the
// row is in use): sa, cu, cv, fu, fv, dbe(r+1); mom: 0 <= r < ny-1 (momentum row),
// in: 0 < r < ny-1 (stage row).
template <typename T>
struct AdjRow {
    T sa, cu, cv, fu, fv, dbe1;
    bool mom, in;
};

template <typename T>
__device__ __forceinline__ AdjRow<T> adj_row(const AdjArgs<T> &a, int r)
{
    const int rc = min(max(r, 0), a.ny - 1);
    AdjRow<T> q;
    q.sa = scalar_load(a.rc.sa + rc);
    q.cu = scalar_load(a.rc.cu + rc);
    q.cv = scalar_load(a.rc.cv + rc);
    q.fu = scalar_load(a.rc.fu + rc);
    q.fv = scalar_load(a.rc.fv + rc);
    q.dbe1 = scalar_load(a.rc.dbe + rc + 1);
    q.mom = r >= 0 && r < a.ny - 1;
    q.in = r > 0 && r < a.ny - 1;
    return q;
}

template <typename T, bool COR, bool EDGE>
__device__ __forceinline__ void adj_march(const AdjArgs<T> &a, int wg, int j0, int j1)
{
    const int lane = threadIdx.x & 63, nx = a.nx, ny = a.ny;
    const int col = wg * kAdjOwn - 1 + lane;             // EDGE: may be -1 or >= nx
    const int ci = EDGE ? min(max(col, 0), nx - 1) : col;
    const bool own = lane >= 1 && lane <= kAdjOwn && (!EDGE || col < nx);
    const bool cmom = !EDGE || (col >= 0 && col < nx - 1), cint = !EDGE || (col > 0 && col < nx - 1);
    const T LF = a.lin_fric_mult, HALF = T(0.5), msl = a.msl;
    const T dle_i = a.rc.dle[EDGE ? min(max(col, 0), nx) : col];
    const T dle_ip1 = a.rc.dle[EDGE ? min(max(col + 1, 0), nx) : col + 1];
    const T mult_i = T(EDGE && col == 0 ? 2 : 1);        // U(0,.) counted twice at i = 0
    struct Row {
        T ls, lu, lv, e;
    };
    auto load_row = [&](int m) {
        const int o = min(EDGE ? max(m, 0) : m, ny - 1) * a.pitch + ci;
        return Row{a.lS[o], a.lU[o], a.lV[o], a.E[o]};
    };
    // of rows m-1, m-2 (m-3): the loaded values, LF l', the pressure terms, the new stage
    // adjoint (as written, and where it is an interior cell's), the Coriolis products
    T ls1 = T(0), lu1 = T(0), lv1 = T(0), e1 = T(0), aU1 = T(0), aUw1 = T(0), mu1 = T(0), pu1 = T(0), puw1 = T(0);
    T aV2 = T(0), oS2 = T(0), in2 = T(0), lu2 = T(0), lv2 = T(0), mu2 = T(0), mv2 = T(0), pu2 = T(0), puw2 = T(0),
      pv2 = T(0), pve2 = T(0), pv3 = T(0), pve3 = T(0);
    AdjRow<T> q1 = adj_row(a, j0 - 2), q2 = q1;
    auto row = [&](const int m, const Row &in, const AdjRow<T> &q0) {
        const T ls0 = in.ls, lu0 = in.lu, lv0 = in.lv, e0 = in.e;
        // row m
        const T hI0 = face_depth(e0, shl1(e0), msl);
        const T mu0 = LF * lu0;
        T aU0 = q0.cu * hI0 * dle_ip1 * mu0;
        if (EDGE) aU0 = (cmom && q0.mom) ? aU0 : T(0);
        const T aUw0 = shr1(aU0);
        // row m-1
        const T hJ1 = face_depth(e1, e0, msl);
        const T mv1 = LF * lv1;
        T aV1 = q1.cv * hJ1 * q1.dbe1 * mv1;
        if (EDGE) aV1 = (cmom && q1.mom) ? aV1 : T(0);
        const T oS1 = (((ls1 + aU1) - aUw1) + aV1) - aV2;
        const T in1 = !EDGE || (cint && q1.in) ? oS1 : T(0);
        T pu0 = T(0), puw0 = T(0), pv1 = T(0), pve1 = T(0);
        if (COR) {
            pu0 = (hI0 > T(0) ? HALF * q0.fu : T(0)) * mu0;
            if (EDGE) pu0 = (cmom && q0.mom) ? pu0 : T(0);
            puw0 = shr1(pu0);
            pv1 = (hJ1 > T(0) ? HALF * q1.fv : T(0)) * mv1;
            if (EDGE) pv1 = (cmom && q1.mom) ? pv1 : T(0);
            pve1 = shl1(pv1);
            if (EDGE) pv1 = mult_i * pv1;
        }
        // row m-2
        const int r = m - 2;
        const bool mom2 = !EDGE || (cmom && q2.mom);
        T lu_o = (mom2 ? mu2 : lu2) - q2.sa * dle_i * in2;
        T lv_o = (mom2 ? mv2 : lv2) - q2.sa * q2.dbe1 * in2;
        lu_o += q2.sa * dle_ip1 * shl1(in2);
        lv_o += q1.sa * q2.dbe1 * in1;
        if (COR) {
            const T mult_j = T(EDGE && r == 0 ? 2 : 1);  // V(.,0) counted twice at j = 0
            lu_o -= (((T(0) + pv2) + pve2) + pv3) + pve3;
            lv_o += (((T(0) + mult_j * pu2) + mult_j * puw2) + pu1) + puw1;
        }
        if (own && r >= j0 && r < j1) {
            const int ow = r * a.pitch + col;
            a.oS[ow] = oS2;
            a.oU[ow] = lu_o;
            a.oV[ow] = lv_o;
        }
        pv3 = pv2; pve3 = pve2;
        aV2 = aV1; oS2 = oS1; in2 = in1; lu2 = lu1; lv2 = lv1; mu2 = mu1; mv2 = mv1;
        pu2 = pu1; puw2 = puw1; pv2 = pv1; pve2 = pve1;
        ls1 = ls0; lu1 = lu0; lv1 = lv0; e1 = e0; aU1 = aU0; aUw1 = aUw0; mu1 = mu0; pu1 = pu0; puw1 = puw0;
        q2 = q1; q1 = q0;
    };
    Row ra = load_row(j0 - 1), rb = load_row(j0);
    AdjRow<T> qa = adj_row(a, j0 - 1), qb = adj_row(a, j0);
    for (int m = j0 - 1; m <= j1 + 1; m += 2) {
        const Row na = load_row(m + 2), nb = load_row(m + 3);
        const AdjRow<T> nqa = adj_row(a, m + 2), nqb = adj_row(a, m + 3);
        row(m, ra, qa);
        row(m + 1, rb, qb);
        ra = na; rb = nb;
        qa = nqa; qb = nqb;
    }
}

template <typename T, bool COR>
__global__ __launch_bounds__(64) void adj_march_kernel(AdjArgs<T> a)
{
    // each XCD takes a contiguous range of strips, whose common rows then meet in its L2
    const unsigned gx = gridDim.x, L = xcd_tile(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
    const int by = (int)(L / gx), wg = (int)(L - (unsigned)by * gx);
    const int c0 = wg * kAdjOwn - 1, j0 = by * a.rows, j1 = min(j0 + a.rows, a.ny);
    // all its columns, and the rows that its strip's results depend on, interior?
    if (c0 >= 1 && c0 + 64 <= a.nx - 2 && j0 >= 2 && j1 + 1 <= a.ny - 2)
        adj_march<T, COR, false>(a, wg, j0, j1);
    else
        adj_march<T, COR, true>(a, wg, j0, j1);
}

// Adds values[g] to lS at the gauge cells: one lane per gauge; the lane of a cell's
// first gauge adds the values of all gauges at that cell in gauge order (the order of
// one-by-one additions), the others skip.
template <typename T>
__global__ void adj_inject_kernel(T *lS, int n, const long long *idx, const double *values)
{
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const long long c = idx[g];
    for (int h = 0; h < g; h++)
        if (idx[h] == c) return;
    T t = lS[c];
    for (int h = g; h < n; h++)
        if (idx[h] == c) t += (T)values[h];
    lS[c] = t;
}

template <typename T, bool COR>
static hipError_t launch_adj_march(const AdjArgs<T> &a0, hipStream_t s)
{
    constexpr int kBlock = 64;
    AdjArgs<T> a = a0;
    if (a.rows <= 0)
        a.rows = fused_rows(a.nx, a.ny, 1, 2, kAdjOwn, 256);
    const int waves = (a.nx + kAdjOwn - 1) / kAdjOwn, wpb = kBlock / 64;
    dim3 grid((waves + wpb - 1) / wpb, (a.ny + a.rows - 1) / a.rows);
    hipLaunchKernelGGL((adj_march_kernel<T, COR>), grid, dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_adjoint_step(const AdjArgs<T> &a, hipStream_t s)
{
    if ((long long)a.pitch * a.ny >= (1LL << 31)) return hipErrorInvalidValue;
    return a.coriolis ? launch_adj_march<T, true>(a, s) : launch_adj_march<T, false>(a, s);
}

template <typename T>
hipError_t launch_adjoint_inject(T *lS, int n, const long long *idx, const double *values, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(adj_inject_kernel<T>, dim3((n + 63) / 64), dim3(64), 0, s, lS, n, idx, values);
    return hipGetLastError();
}

template hipError_t launch_adjoint_step<double>(const AdjArgs<double> &, hipStream_t);
template hipError_t launch_adjoint_step<float>(const AdjArgs<float> &, hipStream_t);
template hipError_t launch_adjoint_inject<double>(double *, int, const long long *, const double *, hipStream_t);
template hipError_t launch_adjoint_inject<float>(float *, int, const long long *, const double *, hipStream_t);

}  // namespace swh
