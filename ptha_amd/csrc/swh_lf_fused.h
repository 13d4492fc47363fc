// Per-cell operations of the leapfrog step and the column-marching kernel that takes several
// steps per launch (batches: swh_leapfrog2.hip; single grids: swh_leapfrog_sg.hip).
#pragma once
#include "swh_bflux.h"
#include "swh_lanes.h"

namespace swh {

namespace {

constexpr int kOwn = 61;   // columns a wavefront of the two-step kernel writes (lanes 1..61)

// Lane shifts across the wavefront (the lane at the open end takes 0).
// Call them on every lane, outside lane-dependent conditions: a lane that does not
// execute the shift leaves the lane reading from it with an undefined value.
template <typename T>
__device__ __forceinline__ T shl1(T v) { return lane_east(v); }   // value of lane + 1
template <typename T>
__device__ __forceinline__ T shr1(T v) { return lane_west(v); }   // value of lane - 1

// Per-row coefficients (uniform across the wavefront), loaded at a clamped row so
// the loads are always in bounds; 'interior' / 'valid' say whether the row updates.
template <typename T>
struct RowCo {
    T sa, cu, cv, fu, fv, dbe_lo, dbe_hi;   // dbe_lo = dbe(j), dbe_hi = dbe(j+1)
    bool interior, valid;                   // stage row (1..ny-2), momentum row (0..ny-2)
};

template <typename T>
__device__ __forceinline__ RowCo<T> row_co(const LFArgs<T> &a, int r)
{
    const int rc = min(max(r, 0), a.ny - 1);
    RowCo<T> q;
    q.sa = a.rc.sa[rc];
    q.cu = a.rc.cu[rc];
    q.cv = a.rc.cv[rc];
    q.fu = a.rc.fu[rc];
    q.fv = a.rc.fv[rc];
    q.dbe_lo = a.rc.dbe[rc];
    q.dbe_hi = a.rc.dbe[rc + 1];
    q.interior = r > 0 && r < a.ny - 1;
    q.valid = r >= 0 && r < a.ny - 1;
    return q;
}

// What the fused kernel carries of a row's coefficients, in scalar registers (a row is the
// same on every lane): those that every level uses again. dbe1 = dbe(r+1) is also dbe of
// the row above.
template <typename T>
struct RowQ {
    T sa, fu, fv, dbe1, cu, cv;   // (cu and cv are used as the row is loaded, where truely linear)
};

template <typename T>
__device__ __forceinline__ RowQ<T> row_q(const LFArgs<T> &a, int r)
{
    const int rc = min(max(r, 0), a.ny - 1);
    return RowQ<T>{scalar_load(a.rc.sa + rc), scalar_load(a.rc.fu + rc),      scalar_load(a.rc.fv + rc),
                   scalar_load(a.rc.dbe + rc + 1), scalar_load(a.rc.cu + rc), scalar_load(a.rc.cv + rc)};
}

// New stage (include.f90:97-113), computed on every lane and kept where the cell
// is interior; no stage boundary in this kernel.
template <typename T, bool KAHAN>
__device__ __forceinline__ void stage_cell(bool interior, T sa, T dle_i, T dbe_lo, T dbe_hi, T s, T c, T uh, T uhm,
                                           T vh, T vhm, T &sn, T &cn)
{
    const T delta = sa * ((uh - uhm) * dle_i + (vh * dbe_hi - vhm * dbe_lo));
    T t, cc;
    if (KAHAN) {
        const T y = -delta - c;
        t = s + y;
        cc = (t - s) - y;
    } else {
        t = s - delta;
        cc = T(0);
    }
    sn = interior ? t : s;
    cn = interior ? cc : c;
}

// Depth at a face of the truely-linear scheme (include.f90:265-280) from the elevations
// of its two cells (e_far: the east or north one); it depends on the elevation alone.
template <typename T>
__device__ __forceinline__ T tl_face_depth(T e_near, T e_far, T msl)
{
    const T MIN = T(kMinDepth), HALF = T(0.5);
    return (e_near < -MIN + msl && e_far < -MIN + msl) ? msl - HALF * (e_far + e_near) : T(0);
}

// UH at (ii + 1/2, j) from the new stage of cells ii, ii+1 and the pre-step VH of
// rows j-1 (vhm0, vhm1 at ii, ii+1) and j (vh0, vh1).
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
__device__ __forceinline__ T mom_u(const LFArgs<T> &a, bool valid, T cu, T fu, T dle_ip1, T fwu, T uh_old, T s0,
                                   T c0, T s1, T c1, T e0, T e1, T vhm0, T vhm1, T vh0, T vh1)
{
    const T MIN = T(kMinDepth), HALF = T(0.5), msl = a.msl;
    T h_iph, wet_iph;
    if (TL) {
        h_iph = tl_face_depth(e0, e1, msl);
        wet_iph = T(1);
    } else {
        h_iph = (s0 - e0 > MIN && s1 - e1 > MIN) ? HALF * ((s1 + s0) - (e1 + e0)) : T(0);
        wet_iph = h_iph > T(0) ? T(1) : T(0);
    }
    T ds_i = s1 - s0;
    if (KAHAN) ds_i = ds_i - (c1 - c0);
    T uh_new = uh_old * wet_iph - cu * h_iph * ds_i * dle_ip1;
    if (COR || FRIC) {
        const T vh_jmh = HALF * (vhm0 + vhm1);
        const T vh_jph = HALF * (vh0 + vh1);
        if (COR) {
            const T dhc = fu * (h_iph > T(0) ? T(1) : T(0));
            uh_new = uh_new + dhc * (vh_jmh + vh_jph);
        }
        if (FRIC) {
            const T vbar = HALF * (vh_jmh + vh_jph);
            const T fmu = T(1) / (T(1) + a.dt_lfc + a.dt * fwu * (sqrt(uh_old * uh_old + vbar * vbar)));
            uh_new = fmu * uh_new;
        }
    }
    if (LINF) uh_new = a.lin_fric_mult * uh_new;
    return valid ? uh_new : uh_old;
}

// VH at (ii, j + 1/2) from the new stage of rows j, j+1 and the pre-step UH of
// row j (uh_i at ii, uh_im1 at ii-1) and row j+1 (uhu_i, uhu_im1).
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF>
__device__ __forceinline__ T mom_v(const LFArgs<T> &a, bool valid, T cv, T fv, T dbe_hi, T fwv, T vh_old, T s0, T c0,
                                   T sup, T cup, T e0, T eu, T uh_i, T uh_im1, T uhu_i, T uhu_im1)
{
    const T MIN = T(kMinDepth), HALF = T(0.5), msl = a.msl;
    T h_jph, wet_jph;
    if (TL) {
        h_jph = tl_face_depth(e0, eu, msl);
        wet_jph = T(1);
    } else {
        h_jph = (sup - eu > MIN && s0 - e0 > MIN) ? HALF * ((sup + s0) - (eu + e0)) : T(0);
        wet_jph = h_jph > T(0) ? T(1) : T(0);
    }
    T ds_j = sup - s0;
    if (KAHAN) ds_j = ds_j - (cup - c0);
    T vh_new = vh_old * wet_jph - cv * h_jph * ds_j * dbe_hi;
    if (COR || FRIC) {
        const T uh_ij = HALF * (uh_i + uh_im1);
        const T uh_ijp1 = HALF * (uhu_i + uhu_im1);
        if (COR) {
            const T dhcj = fv * (h_jph > T(0) ? T(1) : T(0));
            vh_new = vh_new - dhcj * (uh_ij + uh_ijp1);
        }
        if (FRIC) {
            const T ubar = HALF * (uh_ij + uh_ijp1);
            const T fmv = T(1) / (T(1) + a.dt_lfc + a.dt * fwv * (sqrt(vh_old * vh_old + ubar * ubar)));
            vh_new = fmv * vh_new;
        }
    }
    if (LINF) vh_new = a.lin_fric_mult * vh_new;
    return valid ? vh_new : vh_old;
}

}  // namespace

// The tile (column block, strip, source) of this workgroup. Workgroups are dispatched
// to the 8 XCDs (each with its own L2) round-robin by linear index; in XCD order the
// i-th workgroup on an XCD takes the i-th tile of that XCD's contiguous range of tiles,
// ordered columns fastest, then the sources of a group of 'group' sources, then
// strips, then groups. Neighbouring tiles of a strip, the sources of a group (which
// read the same elevation and row coefficients) and the next strip (which reads the
// halo rows of this one) thus run on the same L2 shortly after one another.
// ey: rows of workgroups ahead of the tiles that do other work (single grid only).
__device__ __forceinline__ void lf2_tile(int order, int group, int ey, int &bx, int &by, int &bz)
{
    bx = blockIdx.x; by = (int)blockIdx.y - ey; bz = blockIdx.z;
    if (!order) return;
    const unsigned gx = gridDim.x, gy = gridDim.y - ey, gz = gridDim.z;
    const unsigned B = gx * gy * gz;
    const unsigned b = blockIdx.x + gx * ((blockIdx.y - ey) + gy * blockIdx.z);
    const unsigned L = xcd_tile(b, B);
    const unsigned G = (unsigned)group;
    const unsigned gi = L / (gx * gy * G);                 // source group
    const unsigned within = L - gi * (gx * gy * G);
    const unsigned Gi = min(G, gz - gi * G);               // sources in this group (the last may be short)
    const unsigned t = within / gx;
    bx = (int)(within - t * gx);
    bz = (int)(gi * G + t % Gi);
    by = (int)(t / Gi);
}

// The momentum of one face after a step, from the new stage of its two cells (near, far)
// and the averages am, ap of the other momentum on its two sides (rows j-1/2 and j+1/2 for
// UH, which adds the Coriolis term; rows j and j+1 for VH, which subtracts it): the
// operations of mom_u / mom_v in their order, with what several levels or rows share
// taken out. Truely linear: ch = coefficient * face depth, formed once per row (positive
// where the face is wet); else cg, e_near, e_far give the depth at the new stage.
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, bool U>
__device__ __forceinline__ T mom_face(const LFArgs<T> &a, T ch, T cg, T f, T len, T fw, T old, T s_near, T c_near,
                                      T s_far, T c_far, T e_near, T e_far, T am, T ap)
{
    const T MIN = T(kMinDepth), HALF = T(0.5);
    T x = old;
    if (!TL) {
        const T h = (s_near - e_near > MIN && s_far - e_far > MIN) ? HALF * ((s_far + s_near) - (e_far + e_near)) : T(0);
        x = old * (h > T(0) ? T(1) : T(0));
        ch = cg * h;
    }
    T ds = s_far - s_near;
    if (KAHAN) ds = ds - (c_far - c_near);
    x = x - ch * ds * len;
    if (COR || FRIC) {
        const T sum = am + ap;
        if (COR) {
            const T d = ch > T(0) ? f : T(0);
            x = U ? x + d * sum : x - d * sum;
        }
        if (FRIC) {
            const T bar = HALF * sum;
            const T fm = T(1) / (T(1) + a.dt_lfc + a.dt * fw * (sqrt(old * old + bar * bar)));
            x = fm * x;
        }
    }
    if (LINF) x = a.lin_fric_mult * x;
    return x;
}

// NS fused steps per launch (the state is read and written once per NS steps). The same
// per-cell operations as the one-step kernel, scheduled as in leapfrog2_kernel but for any
// number of levels: at row m, level n (the state after n steps) forms its stage and UH at
// row m-n+1 and its VH at row m-n from level n-1, whose stage and UH of row m-n+1 were
// formed in the previous iteration (level 0: the row loaded now) and whose VH of rows m-n+1
// (this iteration) and m-n (the previous one) are at hand; row m-NS of level NS is written.
// Each level consumes one lane of the wavefront to the west (UH(i-1)) and one to the east
// (stage(i+1), VH(i+1)), so a wavefront owns 65 - 2 NS of its 64 columns; each strip
// recomputes NS rows below and NS - 1 above it.
//
// What bounds it: instructions (a SIMD issues one VALU operation in about 4.5 clocks whatever
// its kind), so everything but the scheme's own operations is taken out of the rows' loop:
//  - INNER: a wavefront whose columns and rows are all interior (nearly every one) runs
//    without the selections of the grid's edges;
//  - the averages that the Coriolis and friction terms take of the other momentum are formed
//    once per row and level and carried to the next row, which needs them again;
//  - coefficient * face depth is formed once per row, not once per level;
//  - neighbour columns are lane shifts that fold into the operation that uses them;
//  - two rows per loop iteration, so that what is carried changes registers by name;
//  - row coefficients come a row ahead through the scalar cache (scalar_load: as vector loads
//    they waited behind the next row's state).
// In FP32 with Coriolis a row of five levels is 245 vector operations (384 before) in the
// INNER loop. Measured per step: 12 sources of 1200 x 1200 in FP32 49 -> 42.5 us, 32 sources
// 123 -> 100, 1 source 7.6 -> 5.8; 512 sources 1.67 -> 1.45 ms. FP64: 12 sources 99 -> 64,
// 1 source 11.3 -> 7.5.
// MX (single grids): max_stage after every step. The running maxima of the NS rows in
// flight move up a ring beside the levels; a row's are read once, before level 1, and
// written once, after level NS.
// EDGE (single grids): a wavefront that may hold a boundary-flux line: the lanes that own it
// store UH or VH of levels 0 to NS-1 (the pre-step values of the launch's steps) to a line
// buffer.
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, bool PF, int NS, bool GS, bool MX, bool EDGE,
          bool INNER>
__device__ __forceinline__ void leapfrogn_march(const LFArgs<T> &a, int bx, int by, int bz)
{
    constexpr int OWN = 65 - 2 * NS;
    const T HALF = T(0.5);
    const int lane = threadIdx.x & 63;
    const int wg = bx * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (wg * OWN >= a.nx) return;                        // whole wavefront past the east edge
    const int col = wg * OWN - (NS - 1) + lane;          // column of this lane (may be < 0 or >= nx)
    const int ci = INNER ? col : min(max(col, 0), a.nx - 1);   // column it loads (clamped into the row)
    const bool own = lane >= NS - 1 && lane < NS - 1 + OWN && col < a.nx;
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
    const bool west = !INNER && col == 0;                // UH(i-1) clamps to UH(0) (include.f90:319-322)
    const T dle_i = a.rc.dle[min(max(col, 0), a.nx)];
    const T dle_ip1 = a.rc.dle[min(max(col + 1, 0), a.nx)];
    const bool col_int = INNER || (col > 0 && col < a.nx - 1);    // stage: interior column
    const bool col_mom = INNER || (col >= 0 && col < a.nx - 1);   // momentum: UH/VH of this column update
    // the gauges in this lane's own column and rows j0..j1-1 (the host sees that there are
    // at most two): indices + 1 in bytes 0 and 1 of gk (0: none), rows in the halves of gr
    int gk = 0, gr = 0;
    if (GS) {
        // each lane looks at one gauge of 64; what lies in this wavefront's tile is rare
        for (int g0 = 0; g0 < a.g_n; g0 += 64) {
            const int g = min(g0 + lane, a.g_n - 1);
            const int gi = a.g_ij[2 * g], gj = a.g_ij[2 * g + 1];
            unsigned long long m = __ballot(g0 + lane < a.g_n && gj >= j0 && gj < j1 && gi >= wg * OWN &&
                                            gi < (wg + 1) * OWN);
            for (; m; m &= m - 1) {
                const int b = __builtin_ctzll(m);
                const int bi = __builtin_amdgcn_readlane(gi, b), bj = __builtin_amdgcn_readlane(gj, b);
                if (own && bi == col) {
                    if (gk == 0) { gk = g0 + b + 1; gr = bj; }
                    else { gk |= (g0 + b + 1) << 8; gr |= bj << 16; }
                }
            }
        }
    }

    // maxima of rows m-k
    T mx_r[NS];
    T *__restrict__ const mxp = MX ? a.mx + (long long)MX_STAGE * a.pitch * a.ny : nullptr;
    // boundary-flux lines: UH of this lane's column (E line 1, W line 3; at 'line', null
    // elsewhere) and VH of two rows (N line 0, S line 2), level l, to the line buffer
    // [level][side][lb_len]; le0..le0+le_n-1 the rows of the columns in this strip
    const int ne = a.bf.n_ext;
    T *line = nullptr;
    if (EDGE && own && (col == a.nx - ne - 1 || col == ne - 1))
        line = a.lb_out + (col == ne - 1 ? 3 : 1) * a.lb_len - ne;
    const bool line_ns = EDGE && own && col >= ne && col < a.nx - ne;
    const int le0 = max(j0, ne), le_n = max(min(j1, a.ny - ne) - le0, 0);
    const int rowN = a.ny - ne - 1 >= j0 && a.ny - ne - 1 < j1 ? a.ny - ne - 1 : -1000000;
    const int rowS = ne - 1 >= j0 && ne - 1 < j1 ? ne - 1 : -1000000;
    auto keep_lines = [&](int l, int ru, T uh, int rv, T vh) {
        if ((unsigned)(ru - le0) < (unsigned)le_n && line) line[4 * l * a.lb_len + ru] = uh;
        if ((rv == rowN || rv == rowS) && line_ns) a.lb_out[(4 * l + (rv == rowS ? 2 : 0)) * a.lb_len + col - ne] = vh;
    };

    // carried between rows, per level n (0 = the loaded state)
    T s_p[NS + 1], c_p[NS + 1];   // stage of level n at its stage row of the previous iteration
    T uh_p[NS + 1];               // its UH there
    T vh_p[NS + 1], va_p[NS + 1]; // its VH of the previous iteration, and its average with the east one
    T ua_p[NS + 1];               // average of level n-1's UH and its west one, a row lower
    // truely linear: coefficient * face depth of UH's row m-k, and of VH's row m-1-k; else the
    // elevation of row m-k and its east value
    T ci_r[NS], cj_r[NS], e_r[NS + 1], e_rr[NS + 1], e_prev = T(0);
    T fwu_r[NS], fwv_r[NS];       // friction work: UH at row m-k, VH at row m-1-k
    RowQ<T> q_r[NS + 1];          // row coefficients of row m-k
#pragma unroll
    for (int n = 0; n <= NS; n++) {
        s_p[n] = T(0); c_p[n] = T(0); uh_p[n] = T(0); vh_p[n] = T(0); va_p[n] = T(0); ua_p[n] = T(0);
        e_r[n] = T(0); e_rr[n] = T(0);
    }
#pragma unroll
    for (int n = 0; n < NS; n++) {
        ci_r[n] = T(0); cj_r[n] = T(0); fwu_r[n] = T(0); fwv_r[n] = T(0); mx_r[n] = T(0);
    }
    const int m0 = j0 - NS + 1;
    // the rings as they stand after row m0-1 (each iteration first slides them by one)
#pragma unroll
    for (int k = 0; k <= NS; k++) q_r[k] = row_q(a, m0 - 1 - k);
    {
        // the row below the first one: pre-step VH/UH/E of row m0-1
        const int o = min(max(m0 - 1, 0), a.ny - 1) * a.pitch + ci;
        vh_p[0] = VH[o];
        va_p[0] = HALF * (vh_p[0] + shl1(vh_p[0]));
        const T uh = UH[o], uh_sh = shr1(uh);
        ua_p[1] = HALF * (uh + (west ? uh : uh_sh));
        e_r[0] = e_prev = a.E[o];
        e_rr[0] = shl1(e_r[0]);
    }
    auto load_row = [&](int m, T &s0, T &c0, T &uh0, T &vh0, T &e, T &uhw, T &fwu, T &fwv) {
        const int mr = min(max(m, 0), a.ny - 1);
        const int o = mr * a.pitch + ci;
        s0 = S[o];
        c0 = KAHAN ? C[o] : T(0);
        uh0 = UH[o];
        vh0 = VH[o];
        e = a.E[o];
        uhw = T(0);
        if (lane == 0 && col > 0) uhw = UH[o - 1];
        fwu = FRIC ? a.fwU[o] : T(0);
        fwv = FRIC ? a.fwV[min(max(m - 1, 0), a.ny - 1) * a.pitch + ci] : T(0);
    };
    // max_stage of the rows this strip owns (0: not needed)
    auto load_mx = [&](int m) {
        return (own && m >= j0 && m < j1) ? mxp[(long long)m * a.pitch + col] : T(0);
    };
    T n_s0, n_c0, n_uh0, n_vh0, n_e, n_uhw, n_fwu, n_fwv, n_mx = T(0);
    if (PF) load_row(m0, n_s0, n_c0, n_uh0, n_vh0, n_e, n_uhw, n_fwu, n_fwv);
    if (MX && PF) n_mx = load_mx(m0);
    RowQ<T> n_q = row_q(a, m0);
    T cap_s = T(0), cap_c = T(0), cap_uh = T(0), cap_vh = T(0);   // the sampled level (gauges)

    auto row = [&](const int m) {
        T s0, c0, uh0, vh0, e0, uhw, fwu, fwv;
        if (PF) {
            s0 = n_s0; c0 = n_c0; uh0 = n_uh0; vh0 = n_vh0; e0 = n_e; uhw = n_uhw;
            fwu = n_fwu; fwv = n_fwv;
            if (MX) {
#pragma unroll
                for (int k = NS - 1; k >= 1; k--) mx_r[k] = mx_r[k - 1];
                mx_r[0] = n_mx;
                n_mx = load_mx(m + 1);
            }
            load_row(m + 1, n_s0, n_c0, n_uh0, n_vh0, n_e, n_uhw, n_fwu, n_fwv);
        } else {
            load_row(m, s0, c0, uh0, vh0, e0, uhw, fwu, fwv);
        }
        // slide the rings of rows: index k now holds row m-k
#pragma unroll
        for (int k = NS; k >= 1; k--) q_r[k] = q_r[k - 1];
        q_r[0] = n_q;
        n_q = row_q(a, m + 1);
        if constexpr (TL) {
#pragma unroll
            for (int k = NS - 1; k >= 1; k--) { ci_r[k] = ci_r[k - 1]; cj_r[k] = cj_r[k - 1]; }
            ci_r[0] = q_r[0].cu * tl_face_depth(e0, shl1(e0), a.msl);
            cj_r[0] = q_r[1].cv * tl_face_depth(e_prev, e0, a.msl);
            e_prev = e0;
        } else {
#pragma unroll
            for (int k = NS; k >= 1; k--) { e_r[k] = e_r[k - 1]; e_rr[k] = e_rr[k - 1]; }
            e_r[0] = e0;
            e_rr[0] = shl1(e0);
        }
        if (FRIC) {
#pragma unroll
            for (int k = NS - 1; k >= 1; k--) { fwu_r[k] = fwu_r[k - 1]; fwv_r[k] = fwv_r[k - 1]; }
            fwu_r[0] = fwu;
            fwv_r[0] = fwv;
        }
        // inputs of the level being formed: stage/UH of the level below at this level's
        // stage row (UH(i-1): the west lane's; of the loaded row, lane 0's from memory), its VH
        // there
        T in_s = s0, in_c = c0, in_uh = uh0, vh_cur = vh0;
        T out_s = T(0), out_c = T(0), out_uh = T(0), out_vh = T(0);
        if (EDGE) keep_lines(0, m, uh0, m, vh0);
#pragma unroll
        for (int n = 1; n <= NS; n++) {
            const int r = m - n + 1;                  // this level's stage/UH row
            const RowQ<T> &q = q_r[n - 1];            // row r
            const RowQ<T> &qb = q_r[n];               // row r-1
            T in_uh_l = n == 1 ? lane_west_or(in_uh, uhw) : shr1(in_uh);
            if (west) in_uh_l = in_uh;
            // VH of the level below at row r-1, clamped to row r at the southern edge
            const T vhb = INNER || r > 0 ? vh_p[n - 1] : vh_cur;
            T sn, cn;
            stage_cell<T, KAHAN>(INNER || (col_int && (unsigned)(r - 1) < (unsigned)(a.ny - 2)), q.sa, dle_i, qb.dbe1, q.dbe1, in_s, in_c, in_uh,
                                 in_uh_l, vh_cur, vhb, sn, cn);
            T va = T(0), vam = T(0), ua = T(0), uam = T(0);
            if (COR || FRIC) {
                va = HALF * (vh_cur + shl1(vh_cur));
                vam = INNER || r > 0 ? va_p[n - 1] : va;
                ua = HALF * (in_uh + in_uh_l);
                uam = ua_p[n];
            }
            T uhn = mom_face<T, KAHAN, COR, FRIC, TL, LINF, true>(
                a, ci_r[n - 1], q.cu, q.fu, dle_ip1, FRIC ? fwu_r[n - 1] : T(0), in_uh, sn, cn, shl1(sn),
                KAHAN ? shl1(cn) : T(0), TL ? T(0) : e_r[n - 1], TL ? T(0) : e_rr[n - 1], vam, va);
            // VH at row r-1: stage of this level at rows r-1 (previous iteration) and r,
            // UH of the level below at rows r-1 and r
            T vhn = mom_face<T, KAHAN, COR, FRIC, TL, LINF, false>(
                a, cj_r[n - 1], qb.cv, qb.fv, qb.dbe1, FRIC ? fwv_r[n - 1] : T(0), vh_p[n - 1], s_p[n], c_p[n], sn, cn,
                TL ? T(0) : e_r[n], TL ? T(0) : e_r[n - 1], uam, ua);
            if (!INNER) {
                uhn = col_mom && (unsigned)r < (unsigned)(a.ny - 1) ? uhn : in_uh;
                vhn = col_mom && (unsigned)(r - 1) < (unsigned)(a.ny - 1) ? vhn : vh_p[n - 1];
            }
            if (MX) {
                // update_max_quantities after step n (domain_mod.f90:2243-2404), as the
                // one-step kernel: the represented stage, a NaN replaces the maximum
                const T st = KAHAN ? sn - cn : sn;
                mx_r[n - 1] = mx_r[n - 1] > st ? mx_r[n - 1] : st;
            }
            if (EDGE && n < NS) keep_lines(n, r, uhn, r - 1, vhn);
            if (GS && n == a.g_level) {
                // the sampled level's values at this iteration's rows
                cap_s = sn; cap_c = cn; cap_uh = uhn; cap_vh = vhn;
            }
            if (n == NS) {
                out_s = s_p[n]; out_c = c_p[n]; out_uh = uh_p[n]; out_vh = vhn;
            }
            // the level below's VH of this iteration becomes its 'previous' one
            vh_p[n - 1] = vh_cur;
            va_p[n - 1] = va;
            ua_p[n] = ua;
            // inputs of level n+1: this level's stage/UH of the previous iteration (row
            // m-n), this level's VH now (row m-n); slide this level
            in_s = s_p[n]; in_c = c_p[n]; in_uh = uh_p[n];
            vh_cur = vhn;
            s_p[n] = sn; c_p[n] = cn; uh_p[n] = uhn;
        }
        if (GS && gk) {
            // the gauge samples after the launch's g_level-th step: stage and UH of row r,
            // VH of row r-1
            const int r = m - a.g_level + 1;
            double *v = a.g_val + ((long long)(bz + a.src_base) * a.g_max + a.g_sample) * 3 * a.g_n;
            const double st = KAHAN ? (double)cap_s - (double)cap_c : (double)cap_s;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int g = ((gk >> (8 * q)) & 255) - 1, row = (gr >> (16 * q)) & 0xffff;
                if (g >= 0 && r == row) { v[g] = st; v[a.g_n + g] = (double)cap_uh; }
                if (g >= 0 && r - 1 == row) v[2 * a.g_n + g] = (double)cap_vh;
            }
        }
        if (MX) {
            const int rm = m - NS + 1;   // level NS's stage row
            if (own && rm >= j0 && rm < j1) mxp[(long long)rm * a.pitch + col] = mx_r[NS - 1];
        }
        const int k = m - NS;
        if (own && k >= j0 && k < j1) {
            const int ow = k * a.pitch + col;
            So[ow] = out_s;
            if (KAHAN) Co[ow] = out_c;
            UHo[ow] = out_uh;
            VHo[ow] = out_vh;
        }
    };
    // (the row past the last one, where their number is odd, writes nothing)
    for (int m = m0; m <= j1 + NS - 1; m += 2) {
        row(m);
        row(m + 1);
    }
}

// Whether the wavefront that owns columns from wg * OWN works on interior cells only: all
// its columns and the rows that its strip's results depend on.
template <int NS>
__device__ __forceinline__ bool lfn_inner(int nx, int ny, int rows, int wg, int by)
{
    const int c0 = wg * (65 - 2 * NS) - (NS - 1), j0 = by * rows, j1 = min(j0 + rows, ny);
    return c0 >= 1 && c0 + 63 <= nx - 2 && j0 - NS >= 1 && j1 + NS <= ny - 1;
}

template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, bool PF, int NS, bool GS = false>
__global__ __launch_bounds__(256, GS && sizeof(T) == 4 ? 4 : 1) void leapfrogn_kernel(LFArgs<T> a)
{
    int bx, by, bz;
    lf2_tile(a.lf2_order, a.lf2_group, 0, bx, by, bz);
    const int wg = __builtin_amdgcn_readfirstlane(bx * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6));
    if (lfn_inner<NS>(a.nx, a.ny, a.rows_per_block, wg, by))
        leapfrogn_march<T, KAHAN, COR, FRIC, TL, LINF, PF, NS, GS, false, false, true>(a, bx, by, bz);
    else
        leapfrogn_march<T, KAHAN, COR, FRIC, TL, LINF, PF, NS, GS, false, false, false>(a, bx, by, bz);
}

}  // namespace swh
