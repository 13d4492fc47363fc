// Several leapfrog steps of a single grid per launch.
//
// What bounds a single grid's step: taken one at a time, a step with its max_stage update
// moves 44 B (FP32K) or 72 B (FP64) per cell and pays a launch; on small grids the launch and
// the latency of one pass over the strips are all of it. Fused steps (leapfrogn_march of
// swh_lf_fused.h, as for batches) read and write the state and the maxima once per launch.
// What a grid keeps between steps is kept inside: max_stage after every step in registers
// beside the levels, and the boundary-flux lines of every level in a small buffer that the
// next launch (or a flush) sums. Measured per step, with max_stage: 400^2 FP64 9.9 -> 4.5 us,
// 2048^2 FP32 50 -> 15, 1201 x 907 FP64 with friction 31 -> 17; without, 1024^2 FP32 8.4 -> 5.6.
// What bounds it now: at 2048^2 about equally the state's trips through the caches and the
// issue of vector operations; at 400^2 the chain of the 8 rows that a strip of three walks
// (0.9 us a row in FP64) and the launch (3 us).
#include "swh_lf_fused.h"
#include "swh_launch.h"

namespace swh {

// boundary-flux sums of the last fused launch of a call
template <typename T>
__global__ __launch_bounds__(256) void bf_flush_kernel(BfLines b, int nx, int ny, const T *lines, int len_max, int levels)
{
    bf_sum_lines<T>(b, nx, ny, lines, len_max, levels, blockIdx.x, gridDim.x);
}

template <typename T>
hipError_t launch_bf_flush(const BfLines &b, int nx, int ny, const T *lines, int len_max, int levels, hipStream_t s)
{
    if (b.want < 4 || b.want > b.cap || levels < 1 || levels > kFusedSteps || !b.part || !b.sc) return hipErrorInvalidValue;
    hipLaunchKernelGGL(bf_flush_kernel<T>, dim3(b.want), dim3(256), 0, s, b, nx, ny, lines, len_max, levels);
    return hipGetLastError();
}
template hipError_t launch_bf_flush<double>(const BfLines &, int, int, const double *, int, int, hipStream_t);
template hipError_t launch_bf_flush<float>(const BfLines &, int, int, const float *, int, int, hipStream_t);

// The first a.bf.ey rows of workgroups take the boundary-flux sums of the launch before
// this one from its line buffer; the others the tiles.
template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, int NS, bool GS, bool MX>
__global__ __launch_bounds__(128) void leapfrog_sg_kernel(LFArgs<T> a)
{
    if ((int)blockIdx.y < a.bf.ey) {
        bf_sum_lines<T>(a.bf, a.nx, a.ny, a.lb_in, a.lb_len, a.lb_levels, (int)(blockIdx.x + gridDim.x * blockIdx.y),
                        (int)gridDim.x * a.bf.ey);
        return;
    }
    int bx, by, bz;
    lf2_tile(a.lf2_order, a.lf2_group, a.bf.ey, bx, by, bz);
    if (GS && a.g_time && bx == 0 && by == 0 && threadIdx.x == 0) *a.g_time = a.g_t;
    // does this wavefront hold a boundary-flux line?
    constexpr int OWN = 65 - 2 * NS;
    const int wg = __builtin_amdgcn_readfirstlane(bx * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6));
    const int ne = a.bf.n_ext, c0 = wg * OWN, r0 = by * a.rows_per_block;
    const auto in = [](int v, int lo, int n) { return v >= lo && v < lo + n; };
    const bool edge = in(ne - 1, c0, OWN) || in(a.nx - ne - 1, c0, OWN) || in(ne - 1, r0, a.rows_per_block) ||
                      in(a.ny - ne - 1, r0, a.rows_per_block);
    if (!edge && lfn_inner<NS>(a.nx, a.ny, a.rows_per_block, wg, by))
        leapfrogn_march<T, KAHAN, COR, FRIC, TL, LINF, true, NS, GS, MX, false, true>(a, bx, by, 0);
    else
        leapfrogn_march<T, KAHAN, COR, FRIC, TL, LINF, true, NS, GS, MX, true, false>(a, bx, by, 0);
}

template <typename T, bool KAHAN, bool COR, int FRIC, bool TL, bool LINF, int NS>
static hipError_t launch_sg(const LFArgs<T> &a0, hipStream_t s)
{
    constexpr int OWN = 65 - 2 * NS, kBlock = 128;
    LFArgs<T> a = a0;
    const int gx = ((a.nx + OWN - 1) / OWN + kBlock / 64 - 1) / (kBlock / 64);
    a.bf.ey = bf_rows(a.bf, gx);
    if (a.bf.ey < 0) return hipErrorInvalidValue;
    if (a.rows_per_block <= 0) a.rows_per_block = fused_rows(a.nx, a.ny, 1, NS, OWN, sizeof(T) == 4 ? 256 : 128);
    const dim3 grid(gx, (a.ny + a.rows_per_block - 1) / a.rows_per_block + a.bf.ey);
#define SWH_SG(GS, MX) \
    hipLaunchKernelGGL((leapfrog_sg_kernel<T, KAHAN, COR, FRIC, TL, LINF, NS, GS, MX>), grid, dim3(kBlock), 0, s, a)
    if (a.g_n && a.g_level >= 1) {
        if constexpr (TL && FRIC == 0) {
            if (a.mx_levels) return hipErrorInvalidValue;
            SWH_SG(true, false);
        } else {
            return hipErrorInvalidValue;
        }
    } else if (a.mx_levels) {
        SWH_SG(false, true);
    } else {
        SWH_SG(false, false);
    }
#undef SWH_SG
    return hipGetLastError();
}

template <typename T, bool KAHAN, bool COR, int NS>
static hipError_t sg_cf(const LFArgs<T> &a, int fric, int tl, int linf, hipStream_t s)
{
    if (fric) return tl ? launch_sg<T, KAHAN, COR, 1, true, false, NS>(a, s) : hipErrorInvalidValue;
    if (tl) return linf ? launch_sg<T, KAHAN, COR, 0, true, true, NS>(a, s)
                        : launch_sg<T, KAHAN, COR, 0, true, false, NS>(a, s);
    return linf ? launch_sg<T, KAHAN, COR, 0, false, true, NS>(a, s)
                : launch_sg<T, KAHAN, COR, 0, false, false, NS>(a, s);
}

template <typename T, bool KAHAN>
hipError_t launch_leapfrog_sg(const LFArgs<T> &a, int coriolis, int friction_mode, int truely_linear,
                              int linear_friction, hipStream_t s)
{
    if (friction_mode > 1 || a.bc_mask || a.src_stride != 0 || a.src_base || (long long)a.pitch * a.ny >= (1LL << 31) ||
        !a.lb_out || a.nx <= 2 * a.bf.n_ext || a.ny <= 2 * a.bf.n_ext || a.lb_len < a.nx - 2 * a.bf.n_ext ||
        a.lb_len < a.ny - 2 * a.bf.n_ext || (a.mx_levels && (!a.mx || a.mx_levels != (1 << kFusedSteps) - 1)) ||
        (a.bf.want && (!a.lb_in || a.lb_levels < 1 || a.lb_levels > kFusedSteps || !a.bf.part || !a.bf.sc)))
        return hipErrorInvalidValue;
    const int linf = (friction_mode == 0) && linear_friction;
    return coriolis ? sg_cf<T, KAHAN, true, kFusedSteps>(a, friction_mode, truely_linear, linf, s)
                    : sg_cf<T, KAHAN, false, kFusedSteps>(a, friction_mode, truely_linear, linf, s);
}

template hipError_t launch_leapfrog_sg<double, false>(const LFArgs<double> &, int, int, int, int, hipStream_t);
template hipError_t launch_leapfrog_sg<float, true>(const LFArgs<float> &, int, int, int, int, hipStream_t);

}  // namespace swh
