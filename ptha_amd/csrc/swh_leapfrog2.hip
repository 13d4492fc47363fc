// Two leapfrog steps per launch (temporal blocking) for batched unit sources.
//
// Each step is exactly the step of domain_mod_linear_solver_include.f90 (stage
// half-step :92-113, UH/VH half-step :211-571 with Coriolis :408-439, friction
// :441-505 and linear drag :550-557), computed with the same operations in the
// same order as the one-step kernel, so two steps here equal two one-step launches
// bit for bit. What changes is the schedule: the state is read from HBM once and
// written once per two steps, halving the traffic per cell-update.
//
// Work split: a wavefront owns 61 consecutive columns and holds 64 (one halo column
// to the west, two to the east; the westmost lane reads its own west neighbour's
// UH from memory); each lane owns one column and marches up a strip of rows. At
// row m it forms step 1 at row m (stage, UH) and m-1 (VH), then step 2 at row m-1
// (stage, UH) and m-2 (VH), and writes row m-2. East/west neighbours come
// from the adjacent lanes (lane moves or permutes, no LDS tile, no barriers); the
// stencil reaches one column each way per step, which the 3 halo lanes cover.
// Rows below/above the strip are recomputed by the strip itself (3 extra rows).
#include <atomic>

#include "swh_lf_fused.h"
#include "swh_launch.h"

namespace swh {

template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
__device__ __forceinline__ void step1_cell(const LFArgs<T> &a, const T *__restrict__ S, const T *__restrict__ C,
                                           const T *__restrict__ UH, const T *__restrict__ VH, int i, int j, T &s_c,
                                           T &c_c, T &uh1, T &vh1);

// PF: the loads of the next row are issued before the current row is computed, so
// their latency overlaps the arithmetic (one row of loads in flight per lane).
// a.bf.ey > 0 (single grid): the first a.bf.ey rows of workgroups take the boundary-flux
// sums of both steps (the second from UH/VH one step ahead on the lines) and write
// nothing else.
// Neighbours come by lane moves, except in FP32 with friction or depths of the moving surface,
// where the permutes suit better (they leave the vector pipe): us a step at 2048 x 2048 with
// permutes / moves, FP32 friction 26.5 / 27.6, FP32 moving depths 18.7 / 19.2, truely linear
// 18.2 / 18.3, FP64 25.7 / 25.0; 400 x 400 FP64 6.2 / 5.9. Row coefficients are vector loads
// here: through the scalar cache (scalar_load) they are waited for in the row that uses them,
// or a row ahead take registers; at 1024 x 1024 in FP64 with friction 15.0 / 16.6 / 18.4 us a
// step as vector loads / scalar / scalar a row ahead. (4096 x 4096 is 3-10 % faster with scalar
// loads.)
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, bool PF>
__global__ __launch_bounds__(256) void leapfrog2_kernel(LFArgs<T> a)
{
    if (a.bf.ey && (int)blockIdx.y < a.bf.ey) {
        bf_lines<T, 2>(a.bf, a.nx, a.ny, a.pitch, a.UH, a.VH, [&](int i, int j, T &uh1, T &vh1) {
            T s_c, c_c;
            step1_cell<T, KAHAN, COR, FRIC, TL, LINF>(a, a.S, a.C, a.UH, a.VH, i, j, s_c, c_c, uh1, vh1);
        });
        return;
    }
    constexpr bool kMoves = sizeof(T) == 8 || (TL && !FRIC);   // neighbours by lane moves (else permutes)
    int bx, by, bz;
    lf2_tile(a.lf2_order, a.lf2_group, a.bf.ey, bx, by, bz);
    const int lane = threadIdx.x & 63;
    const int wg = bx * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (wg * kOwn >= a.nx) return;                       // whole wavefront past the east edge
    const int col = wg * kOwn - 1 + lane;                // column of this lane (may be -1 or >= nx)
    const int ci = min(max(col, 0), a.nx - 1);           // column it loads (clamped into the row)
    const bool own = lane >= 1 && lane <= kOwn && col < a.nx;
    const int j0 = by * a.rows_per_block;
    if (j0 >= a.ny) return;
    const int j1 = min(j0 + a.rows_per_block, a.ny);
    const long long so = (long long)(bz + a.src_base) * a.src_stride;
    const T *__restrict__ S = a.S + so;
    const T *__restrict__ C = KAHAN ? a.C + so : nullptr;
    const T *__restrict__ UH = a.UH + so;
    const T *__restrict__ VH = a.VH + so;
    T *__restrict__ So = a.So + so;
    T *__restrict__ Co = KAHAN ? a.Co + so : nullptr;
    T *__restrict__ UHo = a.UHo + so;
    T *__restrict__ VHo = a.VHo + so;
    const auto east = [](T v) { if constexpr (kMoves) return shl1(v); else return __shfl_down(v, 1); };
    const auto west_of = [](T v) { if constexpr (kMoves) return shr1(v); else return __shfl_up(v, 1); };
    const bool west = col == 0;                          // UH(i-1) clamps to UH(0) (include.f90:319-322)
    // per-lane constants: edge lengths and where the column updates
    const T dle_i = a.rc.dle[min(max(col, 0), a.nx)];
    const T dle_ip1 = a.rc.dle[min(max(col + 1, 0), a.nx)];
    const bool col_int = col > 0 && col < a.nx - 1;      // stage: interior column
    const bool col_mom = col >= 0 && col < a.nx - 1;     // momentum: UH/VH of this column update
    const int cf = min(max(col, 0), a.nx - 1);           // friction-work column

    // registers carried between rows (named by the row they belong to, relative to m)
    T vh0_p = T(0), vh0_p_r = T(0), uh0_p = T(0), uh0_p_l = T(0), e_p = T(0), e_p_r = T(0), e_pp = T(0);
    T s1_p = T(0), c1_p = T(0);
    T uh1_p = T(0), uh1_p_l = T(0), uh1_pp = T(0), uh1_pp_l = T(0);
    T vh1_pp = T(0), vh1_pp_r = T(0);
    T s2_p = T(0), c2_p = T(0), uh2_p = T(0);
    RowCo<T> q_p = row_co(a, j0 - 2), q_pp = row_co(a, j0 - 3);
    T fw_u_p = T(0), fw_v_p = T(0);
    {
        // pre-step VH/UH/E of row j0-2 (feeds only rows the strip does not write)
        const int r = min(max(j0 - 2, 0), a.ny - 1);
        const int o = r * a.pitch + ci;
        vh0_p = VH[o];
        uh0_p = UH[o];
        e_p = a.E[o];
        vh0_p_r = east(vh0_p);
        // every lane takes part in a shuffle (a lane that skips it leaves its neighbour
        // reading an inactive lane), then the western edge keeps its own value
        const T uh0_p_sh = west_of(uh0_p);
        uh0_p_l = west ? uh0_p : uh0_p_sh;
        e_p_r = east(e_p);
    }

    // the loads of one row (lane 0 also reads its own west neighbour's UH)
    auto load_row = [&](int m, T &s0, T &c0, T &uh0, T &vh0, T &e, T &uhw) {
        const int mr = min(max(m, 0), a.ny - 1);
        const int o = mr * a.pitch + ci;
        s0 = S[o];
        c0 = KAHAN ? C[o] : T(0);
        uh0 = UH[o];
        vh0 = VH[o];
        e = a.E[o];
        uhw = (lane == 0 && col > 0) ? UH[o - 1] : uh0;
    };
    T n_s0, n_c0, n_uh0, n_vh0, n_e, n_uhw;
    if (PF) load_row(j0 - 1, n_s0, n_c0, n_uh0, n_vh0, n_e, n_uhw);

    // offsets within one source's plane fit in 32 bits (uniform base + per-lane offset)
    for (int m = j0 - 1; m <= j1 + 1; m++) {
        const int mr = min(max(m, 0), a.ny - 1);
        T s0, c0, uh0, vh0, e, uh0_mem;
        if (PF) {
            s0 = n_s0; c0 = n_c0; uh0 = n_uh0; vh0 = n_vh0; e = n_e; uh0_mem = n_uhw;
            if (m + 1 <= j1 + 1) load_row(m + 1, n_s0, n_c0, n_uh0, n_vh0, n_e, n_uhw);
        } else {
            load_row(m, s0, c0, uh0, vh0, e, uh0_mem);
        }
        const RowCo<T> q = row_co(a, m);
        // UH(i-1): from the lane to the west; lane 0 has none and reads it itself
        const T uh0_sh = west_of(uh0);
        const T uh0_l = west ? uh0 : (lane == 0 ? uh0_mem : uh0_sh);
        const T vh0_r = east(vh0), e_r = east(e);
        // VH of the row below, clamped to row 0 at the southern edge (include.f90:295-308)
        const T vhb = m > 0 ? vh0_p : vh0, vhb_r = m > 0 ? vh0_p_r : vh0_r;
        // friction work: UH at row m (and m-1 from the last row), VH at row m-1 (and m-2)
        T fw_u1 = T(0), fw_v1 = T(0);
        if (FRIC) {
            fw_u1 = a.fwU[mr * a.pitch + cf];
            fw_v1 = a.fwV[min(max(m - 1, 0), a.ny - 1) * a.pitch + cf];
        }
        const T fw_u2 = fw_u_p, fw_v2 = fw_v_p;

        // step 1: stage and UH at row m
        T s1, c1;
        stage_cell<T, KAHAN>(col_int && q.interior, q.sa, dle_i, q.dbe_lo, q.dbe_hi, s0, c0, uh0, uh0_l, vh0, vhb, s1,
                             c1);
        const T s1_r = east(s1);
        const T c1_r = KAHAN ? east(c1) : T(0);
        const T uh1 = mom_u<T, KAHAN, COR, FRIC, TL, LINF>(a, col_mom && q.valid, q.cu, q.fu, dle_ip1, fw_u1, uh0, s1,
                                                            c1, s1_r, c1_r, e, e_r, vhb, vhb_r, vh0, vh0_r);
        const T uh1_sh = west_of(uh1);
        const T uh1_l = west ? uh1 : uh1_sh;
        // step 1: VH at row m-1
        const T vh1 = mom_v<T, KAHAN, COR, FRIC, TL, LINF>(a, col_mom && q_p.valid, q_p.cv, q_p.fv, q_p.dbe_hi, fw_v1,
                                                            vh0_p, s1_p, c1_p, s1, c1, e_p, e, uh0_p, uh0_p_l, uh0,
                                                            uh0_l);
        const T vh1_r = east(vh1);
        // step 2: stage and UH at row m-1 (VH of row m-2 clamped to row 0 at the southern edge)
        const T vhb1 = m - 1 > 0 ? vh1_pp : vh1, vhb1_r = m - 1 > 0 ? vh1_pp_r : vh1_r;
        T s2, c2;
        stage_cell<T, KAHAN>(col_int && q_p.interior, q_p.sa, dle_i, q_p.dbe_lo, q_p.dbe_hi, s1_p, c1_p, uh1_p,
                             uh1_p_l, vh1, vhb1, s2, c2);
        const T s2_r = east(s2);
        const T c2_r = KAHAN ? east(c2) : T(0);
        const T uh2 = mom_u<T, KAHAN, COR, FRIC, TL, LINF>(a, col_mom && q_p.valid, q_p.cu, q_p.fu, dle_ip1, fw_u2,
                                                            uh1_p, s2, c2, s2_r, c2_r, e_p, e_p_r, vhb1, vhb1_r, vh1,
                                                            vh1_r);
        // step 2: VH at row m-2
        const T vh2 = mom_v<T, KAHAN, COR, FRIC, TL, LINF>(a, col_mom && q_pp.valid, q_pp.cv, q_pp.fv, q_pp.dbe_hi,
                                                            fw_v2, vh1_pp, s2_p, c2_p, s2, c2, e_pp, e_p, uh1_pp,
                                                            uh1_pp_l, uh1_p, uh1_p_l);
        const int k = m - 2;
        if (own && k >= j0 && k < j1) {
            const int ow = k * a.pitch + col;
            So[ow] = s2_p;
            if (KAHAN) Co[ow] = c2_p;
            UHo[ow] = uh2_p;
            VHo[ow] = vh2;
        }
        // slide up one row
        s2_p = s2; c2_p = c2; uh2_p = uh2;
        uh1_pp = uh1_p; uh1_pp_l = uh1_p_l; uh1_p = uh1; uh1_p_l = uh1_l;
        vh1_pp = vh1; vh1_pp_r = vh1_r;
        s1_p = s1; c1_p = c1;
        vh0_p = vh0; vh0_p_r = vh0_r; uh0_p = uh0; uh0_p_l = uh0_l;
        e_pp = e_p; e_p = e; e_p_r = e_r;
        q_pp = q_p; q_p = q;
        fw_u_p = fw_u1; fw_v_p = fw_v1;
    }
}

// One step ahead at one cell: [stage (S, C), UH, VH] after one step at (i, j),
// computed from the state (S, C, UH, VH) with the same per-cell operations as the step
// kernels.
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
__device__ __forceinline__ void step1_cell(const LFArgs<T> &a, const T *__restrict__ S, const T *__restrict__ C,
                                           const T *__restrict__ UH, const T *__restrict__ VH, int i, int j, T &s_c,
                                           T &c_c, T &uh1, T &vh1)
{
    const T *__restrict__ E = a.E;
    const int ip = min(i + 1, a.nx - 1), im = max(i - 1, 0), jp = min(j + 1, a.ny - 1), jm = max(j - 1, 0);
    auto at = [&](int ii, int jj) { return (long long)jj * a.pitch + ii; };
    auto cval = [&](long long o) { return KAHAN ? C[o] : T(0); };
    // VH of the row below, clamped to row 0 at the southern edge
    const T vhb_i = j > 0 ? VH[at(i, jm)] : VH[at(i, j)];
    const T vhb_ip = j > 0 ? VH[at(ip, jm)] : VH[at(ip, j)];
    const RowCo<T> q = row_co(a, j), qu = row_co(a, jp);
    const T dle_i = a.rc.dle[i], dle_ip = a.rc.dle[ip], dle_ip1 = a.rc.dle[i + 1];
    const bool ci_int = i > 0 && i < a.nx - 1, cip_int = ip > 0 && ip < a.nx - 1;
    // new stage at (i, j), (i+1, j), (i, j+1); UH(i-1) clamps to UH(0) at the west edge
    T s_e, c_e, s_n, c_n;
    {
        const long long o = at(i, j);
        stage_cell<T, KAHAN>(ci_int && q.interior, q.sa, dle_i, q.dbe_lo, q.dbe_hi, S[o], cval(o), UH[o],
                             UH[at(im, j)], VH[o], vhb_i, s_c, c_c);
    }
    {
        const long long o = at(ip, j);
        stage_cell<T, KAHAN>(cip_int && q.interior, q.sa, dle_ip, q.dbe_lo, q.dbe_hi, S[o], cval(o), UH[o],
                             UH[at(i, j)], VH[o], vhb_ip, s_e, c_e);
    }
    {
        const long long o = at(i, jp);
        stage_cell<T, KAHAN>(ci_int && qu.interior, qu.sa, dle_i, qu.dbe_lo, qu.dbe_hi, S[o], cval(o), UH[o],
                             UH[at(im, jp)], VH[o], VH[at(i, j)], s_n, c_n);
    }
    const bool mom = i < a.nx - 1 && q.valid;
    const T fwu = FRIC ? a.fwU[at(i, j)] : T(0), fwv = FRIC ? a.fwV[at(i, j)] : T(0);
    uh1 = mom_u<T, KAHAN, COR, FRIC, TL, LINF>(a, mom, q.cu, q.fu, dle_ip1, fwu, UH[at(i, j)], s_c, c_c, s_e, c_e,
                                               E[at(i, j)], E[at(ip, j)], vhb_i, vhb_ip, VH[at(i, j)],
                                               VH[at(ip, j)]);
    vh1 = mom_v<T, KAHAN, COR, FRIC, TL, LINF>(a, mom, q.cv, q.fv, q.dbe_hi, fwv, VH[at(i, j)], s_c, c_c, s_n, c_n,
                                               E[at(i, j)], E[at(i, jp)], UH[at(i, j)], UH[at(im, j)],
                                               UH[at(i, jp)], UH[at(im, jp)]);
}

// Gauge values one step ahead (so a two-step launch can pass over a sampling step).
// One lane per (gauge, source); values[((slot * gmax + sample) * 3 + var) * n + g];
// times (single grid, or null): times[sample] = t.
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
__global__ __launch_bounds__(64) void gauge_step1_kernel(LFArgs<T> a, int n, const long long *__restrict__ idx,
                                                         double *values, int gmax, int sample, double *times,
                                                         double t)
{
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (times && g == 0 && blockIdx.y == 0) times[sample] = t;
    if (g >= n) return;
    const int slot = blockIdx.y + a.src_base;
    const long long so = (long long)slot * a.src_stride;
    const int i = (int)(idx[g] % a.pitch), j = (int)(idx[g] / a.pitch);
    T s_c, c_c, uh1, vh1;
    step1_cell<T, KAHAN, COR, FRIC, TL, LINF>(a, a.S + so, KAHAN ? a.C + so : nullptr, a.UH + so, a.VH + so, i, j,
                                              s_c, c_c, uh1, vh1);
    double *v = values + ((long long)slot * gmax + sample) * 3 * n;
    v[g] = KAHAN ? (double)s_c - (double)c_c : (double)s_c;
    v[n + g] = (double)uh1;
    v[2 * n + g] = (double)vh1;
}

template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
static hipError_t launch_g1(const LFArgs<T> &a, int nsrc, int n, const long long *idx, double *values, int gmax,
                            int sample, double *times, double t, hipStream_t s)
{
    hipLaunchKernelGGL((gauge_step1_kernel<T, KAHAN, COR, FRIC, TL, LINF>), dim3((n + 63) / 64, nsrc), dim3(64), 0, s,
                       a, n, idx, values, gmax, sample, times, t);
    return hipGetLastError();
}

template <typename T, bool KAHAN, bool COR, int FRIC>
static hipError_t g1_tl(const LFArgs<T> &a, int tl, int linf, int nsrc, int n, const long long *idx, double *values,
                        int gmax, int sample, double *times, double t, hipStream_t s)
{
    if (tl)
        return linf ? launch_g1<T, KAHAN, COR, FRIC, true, true>(a, nsrc, n, idx, values, gmax, sample, times, t, s)
                    : launch_g1<T, KAHAN, COR, FRIC, true, false>(a, nsrc, n, idx, values, gmax, sample, times, t, s);
    return linf ? launch_g1<T, KAHAN, COR, FRIC, false, true>(a, nsrc, n, idx, values, gmax, sample, times, t, s)
                : launch_g1<T, KAHAN, COR, FRIC, false, false>(a, nsrc, n, idx, values, gmax, sample, times, t, s);
}

template <typename T, bool KAHAN>
hipError_t launch_gauge_step1(const LFArgs<T> &a, int coriolis, int friction_mode, int truely_linear,
                              int linear_friction, int nsrc, int n, const long long *idx, double *values, int gmax,
                              int sample, double *times, double t, hipStream_t s)
{
    if (friction_mode > 1 || a.bc_mask || n <= 0 || nsrc <= 0) return hipErrorInvalidValue;
    const int linf = (friction_mode == 0) && linear_friction;
    if (coriolis) {
        return friction_mode
                   ? g1_tl<T, KAHAN, true, 1>(a, truely_linear, linf, nsrc, n, idx, values, gmax, sample, times, t, s)
                   : g1_tl<T, KAHAN, true, 0>(a, truely_linear, linf, nsrc, n, idx, values, gmax, sample, times, t, s);
    }
    return friction_mode
               ? g1_tl<T, KAHAN, false, 1>(a, truely_linear, linf, nsrc, n, idx, values, gmax, sample, times, t, s)
               : g1_tl<T, KAHAN, false, 0>(a, truely_linear, linf, nsrc, n, idx, values, gmax, sample, times, t, s);
}

template hipError_t launch_gauge_step1<double, false>(const LFArgs<double> &, int, int, int, int, int, int,
                                                      const long long *, double *, int, int, double *, double,
                                                      hipStream_t);
template hipError_t launch_gauge_step1<float, true>(const LFArgs<float> &, int, int, int, int, int, int,
                                                    const long long *, double *, int, int, double *, double,
                                                    hipStream_t);

// Rows per strip of a single grid when the caller leaves them open (rows_per_block <= 0):
// see occupancy_rows. Measured on a 2048 x 2048 grid: 12-16 rows for the FP32 kernel, 24
// for the FP64 one, against 32 for a fixed 2048-wavefront target.
template <typename K>
static int lf2_auto_rows(K kernel, int nx, int ny, int block_x)
{
    static std::atomic<int> occ[5];   // workgroups per CU, by block_x / 64
    return occupancy_rows((const void *)kernel, occ, nx, ny, block_x, kOwn, 3);
}

template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
static hipError_t launch_lf2(const LFArgs<T> &a0, int nsrc, int block_x, hipStream_t s, int pf)
{
    const int waves = (a0.nx + kOwn - 1) / kOwn, wpb = block_x / 64;
    const int gx = (waves + wpb - 1) / wpb;
    LFArgs<T> a = a0;
    a.bf.ey = bf_rows(a.bf, gx);
    if (a.bf.ey < 0) return hipErrorInvalidValue;
    if (a.rows_per_block <= 0) {
        if (nsrc != 1) return hipErrorInvalidValue;
        a.rows_per_block = pf ? lf2_auto_rows(leapfrog2_kernel<T, KAHAN, COR, FRIC, TL, LINF, true>, a.nx, a.ny,
                                              block_x)
                              : lf2_auto_rows(leapfrog2_kernel<T, KAHAN, COR, FRIC, TL, LINF, false>, a.nx, a.ny,
                                              block_x);
    }
    dim3 grid(gx, (a.ny + a.rows_per_block - 1) / a.rows_per_block + a.bf.ey, nsrc);
    if (pf)
        hipLaunchKernelGGL((leapfrog2_kernel<T, KAHAN, COR, FRIC, TL, LINF, true>), grid, dim3(block_x), 0, s, a);
    else
        hipLaunchKernelGGL((leapfrog2_kernel<T, KAHAN, COR, FRIC, TL, LINF, false>), grid, dim3(block_x), 0, s, a);
    return hipGetLastError();
}

template <typename T, bool KAHAN, bool COR, int FRIC>
static hipError_t lf2_tl(const LFArgs<T> &a, int tl, int linf, int nsrc, int bx, hipStream_t s, int pf)
{
    if (tl) return linf ? launch_lf2<T, KAHAN, COR, FRIC, true, true>(a, nsrc, bx, s, pf)
                        : launch_lf2<T, KAHAN, COR, FRIC, true, false>(a, nsrc, bx, s, pf);
    return linf ? launch_lf2<T, KAHAN, COR, FRIC, false, true>(a, nsrc, bx, s, pf)
                : launch_lf2<T, KAHAN, COR, FRIC, false, false>(a, nsrc, bx, s, pf);
}

template <typename T, bool KAHAN>
hipError_t launch_leapfrog2(const LFArgs<T> &a, int coriolis, int friction_mode, int truely_linear,
                            int linear_friction, int nsrc, int block_x, hipStream_t s, int pf)
{
    if (friction_mode > 1 || a.bc_mask || a.maxq_mask || (block_x % 64) || block_x < 64 || block_x > 256 ||
        (long long)a.pitch * a.ny >= (1LL << 31) ||
        (a.bf.want && (nsrc != 1 || a.src_stride != 0 || !a.bf.part || !a.bf.sc)))
        return hipErrorInvalidValue;
    const int linf = (friction_mode == 0) && linear_friction;
    if (coriolis) {
        return friction_mode ? lf2_tl<T, KAHAN, true, 1>(a, truely_linear, linf, nsrc, block_x, s, pf)
                             : lf2_tl<T, KAHAN, true, 0>(a, truely_linear, linf, nsrc, block_x, s, pf);
    }
    return friction_mode ? lf2_tl<T, KAHAN, false, 1>(a, truely_linear, linf, nsrc, block_x, s, pf)
                         : lf2_tl<T, KAHAN, false, 0>(a, truely_linear, linf, nsrc, block_x, s, pf);
}

template hipError_t launch_leapfrog2<double, false>(const LFArgs<double> &, int, int, int, int, int, int, hipStream_t,
                                                    int);

template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, int NS>
static hipError_t launch_lfn(const LFArgs<T> &a, int nsrc, int block_x, hipStream_t s, int pf)
{
    constexpr int OWN = 65 - 2 * NS;
    const int waves = (a.nx + OWN - 1) / OWN, wpb = block_x / 64;
    dim3 grid((waves + wpb - 1) / wpb, (a.ny + a.rows_per_block - 1) / a.rows_per_block, nsrc);
    if (a.g_n && a.g_level >= 1 && a.g_level <= NS)
        // the variant that writes the gauge samples falling inside the launch (with the
        // next row's loads in flight): used only by launches that hold a sample
        hipLaunchKernelGGL((leapfrogn_kernel<T, KAHAN, COR, FRIC, TL, LINF, true, NS, true>), grid, dim3(block_x), 0, s,
                           a);
    else if (pf)
        hipLaunchKernelGGL((leapfrogn_kernel<T, KAHAN, COR, FRIC, TL, LINF, true, NS>), grid, dim3(block_x), 0, s, a);
    else
        hipLaunchKernelGGL((leapfrogn_kernel<T, KAHAN, COR, FRIC, TL, LINF, false, NS>), grid, dim3(block_x), 0, s, a);
    return hipGetLastError();
}

template <typename T, bool KAHAN, bool COR, int FRIC, int NS>
static hipError_t lfn_tl(const LFArgs<T> &a, int tl, int linf, int nsrc, int bx, hipStream_t s, int pf)
{
    if (tl) return linf ? launch_lfn<T, KAHAN, COR, FRIC, true, true, NS>(a, nsrc, bx, s, pf)
                        : launch_lfn<T, KAHAN, COR, FRIC, true, false, NS>(a, nsrc, bx, s, pf);
    return linf ? launch_lfn<T, KAHAN, COR, FRIC, false, true, NS>(a, nsrc, bx, s, pf)
                : launch_lfn<T, KAHAN, COR, FRIC, false, false, NS>(a, nsrc, bx, s, pf);
}

template <typename T, bool KAHAN, int NS>
static hipError_t lfn_cf(const LFArgs<T> &a, int coriolis, int friction_mode, int tl, int linf, int nsrc, int bx,
                         hipStream_t s, int pf)
{
    if (coriolis)
        return friction_mode ? lfn_tl<T, KAHAN, true, 1, NS>(a, tl, linf, nsrc, bx, s, pf)
                             : lfn_tl<T, KAHAN, true, 0, NS>(a, tl, linf, nsrc, bx, s, pf);
    return friction_mode ? lfn_tl<T, KAHAN, false, 1, NS>(a, tl, linf, nsrc, bx, s, pf)
                         : lfn_tl<T, KAHAN, false, 0, NS>(a, tl, linf, nsrc, bx, s, pf);
}

template <typename T, bool KAHAN>
hipError_t launch_leapfrogn(const LFArgs<T> &a, int coriolis, int friction_mode, int truely_linear,
                            int linear_friction, int nsrc, int block_x, hipStream_t s, int pf, int ns)
{
    if (friction_mode > 1 || a.bc_mask || a.maxq_mask || (block_x % 64) || block_x < 64 || block_x > 256 ||
        (long long)a.pitch * a.ny >= (1LL << 31) || ns < 3 || ns > 6)
        return hipErrorInvalidValue;
    const int linf = (friction_mode == 0) && linear_friction;
    switch (ns) {
    case 3: return lfn_cf<T, KAHAN, 3>(a, coriolis, friction_mode, truely_linear, linf, nsrc, block_x, s, pf);
    case 4: return lfn_cf<T, KAHAN, 4>(a, coriolis, friction_mode, truely_linear, linf, nsrc, block_x, s, pf);
    case 5: return lfn_cf<T, KAHAN, 5>(a, coriolis, friction_mode, truely_linear, linf, nsrc, block_x, s, pf);
    default: return lfn_cf<T, KAHAN, 6>(a, coriolis, friction_mode, truely_linear, linf, nsrc, block_x, s, pf);
    }
}

template hipError_t launch_leapfrogn<double, false>(const LFArgs<double> &, int, int, int, int, int, int, hipStream_t,
                                                    int, int);
template hipError_t launch_leapfrog2<float, true>(const LFArgs<float> &, int, int, int, int, int, int, hipStream_t,
                                                  int);
template hipError_t launch_leapfrogn<float, true>(const LFArgs<float> &, int, int, int, int, int, int, hipStream_t,
                                                  int, int);

}  // namespace swh
