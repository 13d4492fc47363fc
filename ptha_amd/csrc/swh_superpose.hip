// Earthquake events from unit-source gauge series on the FP64 matrix cores.
//
// The reference combines unit-source tsunami time series into events on the host
// (R/examples/austptha_template/SOURCE_ZONES/TEMPLATE/TSUNAMI_EVENTS/
// sum_tsunami_unit_sources.R:555-711, make_tsunami_event_from_unit_sources): for every
// event, the flow series of its unit sources are summed with weight 1 and scaled by
// the event slip (uniform slip), or summed with per-source slips (stochastic slip);
// the stage has msl subtracted before the sum and added back after it. Here the
// series stay where the batched solver wrote them ([slot][sample][3][gauge], FP64)
// and every event of a call is one row of a dense weight matrix W (events x slots),
// so the whole set of events is one product W * X on v_mfma_f64_16x16x4f64, with
// the event's scale/offset and (optionally) the maximum over time of the stage fused
// into the epilogue, which is what a hazard summary keeps per gauge.
#include <algorithm>

#include "swh_internal.h"
#include "swh_rules.h"

namespace swh {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTE = kSupTE;   // events per block tile (2 x 2 waves of 32 x 32)
constexpr int kTN = kSupTN;   // columns per block tile

// seen: a value that *p has held
__device__ __forceinline__ void atomic_max_f64(double *p, double v, double seen)
{
    unsigned long long *q = reinterpret_cast<unsigned long long *>(p);
    unsigned long long old = (unsigned long long)__double_as_longlong(seen);
    while (__longlong_as_double((long long)old) < v) {
        const unsigned long long assumed = old;
        old = atomicCAS(q, assumed, (unsigned long long)__double_as_longlong(v));
        if (old == assumed) break;
    }
}

// MODE 0: out[e][n] for every column n = (sample * 3 + var) * ng + gauge.
// MODE 1: out[e][g] = max over samples s < nvalid[e] of the event's stage at gauge g
//         (blockIdx.z walks chunks of samples; out starts at -inf).
//
// MFMA operand layout (16 x 16 x 4, FP64): lane l supplies A[l % 16][l / 16] (event
// row, source) and B[l / 16][l % 16] (source, column) and holds D[l / 16 + 4 r][l % 16]
// in accumulator element r (checked on gfx950 with a probe of known operands).
template <int MODE, bool FLAG>
__global__ __launch_bounds__(256) void superpose_kernel(SupArgs a)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int e_base = blockIdx.y * kTE + (wave >> 1) * 32;
    const int c_base = blockIdx.x * kTN + (wave & 1) * 32;
    const long long N = (long long)a.gmax * 3 * a.ng;
    const int ncols = MODE == 0 ? (int)N : a.ng;
    // this lane's B columns (two 16-column tiles)
    long long caddr[2];
    bool cok[2];
    double csub[2];
    for (int tj = 0; tj < 2; tj++) {
        const int c = c_base + tj * 16 + li;
        cok[tj] = c < ncols;
        caddr[tj] = cok[tj] ? c : 0;
        const int var = MODE == 0 ? (int)((caddr[tj] / a.ng) % 3) : 0;
        csub[tj] = var == 0 ? a.msl : 0.0;   // stage - msl is linear
    }
    // this lane's A rows (W is zero padded to a multiple of kTE rows and 4 columns)
    const double *w0 = a.W + (long long)(e_base + li) * a.Kpad + lk;
    const double *w1 = w0 + 16LL * a.Kpad;
    const double *m0 = FLAG ? a.M + (long long)(e_base + li) * a.Kpad + lk : nullptr;
    const double *m1 = FLAG ? m0 + 16LL * a.Kpad : nullptr;
    // epilogue rows of this lane: e = e_base + ti * 16 + lk + 4 * r
    double scale[2][4], offs[2][2][4];
    int nval[2][4];
    for (int ti = 0; ti < 2; ti++)
        for (int r = 0; r < 4; r++) {
            const int e = e_base + ti * 16 + lk + 4 * r;
            scale[ti][r] = a.scale[e];
            nval[ti][r] = a.nvalid[e];
            for (int tj = 0; tj < 2; tj++) offs[ti][tj][r] = csub[tj];
        }

    const int s_lo = MODE == 1 ? blockIdx.z * a.s_chunk : 0;
    const int s_hi = MODE == 1 ? min(s_lo + a.s_chunk, a.s_max) : 1;
    double mx[2][2][4];
    bool nan_seen[2][2][4];
    for (int ti = 0; ti < 2; ti++)
        for (int tj = 0; tj < 2; tj++)
            for (int r = 0; r < 4; r++) {
                mx[ti][tj][r] = -__builtin_huge_val();
                nan_seen[ti][tj][r] = false;
            }

    for (int s = s_lo; s < s_hi; s++) {
        const long long soff = MODE == 1 ? (long long)s * 3 * a.ng : 0;
        d4 acc[2][2], accf[2][2];
        for (int ti = 0; ti < 2; ti++)
            for (int tj = 0; tj < 2; tj++) {
                acc[ti][tj] = d4{0.0, 0.0, 0.0, 0.0};
                accf[ti][tj] = d4{0.0, 0.0, 0.0, 0.0};
            }
        const double *xk = a.X + (long long)lk * a.slot_stride + soff;
        for (int k0 = 0; k0 < a.Kpad; k0 += 4) {
            const bool kok = k0 + lk < a.nsrc;
            const double a0 = w0[k0], a1 = w1[k0];
            double b[2], bf[2];
            for (int tj = 0; tj < 2; tj++) {
                b[tj] = (kok && cok[tj]) ? xk[caddr[tj]] - csub[tj] : 0.0;
                if (FLAG) {
                    // a non-finite value enters as 0 (so 0 weights of other events stay 0)
                    // and is counted in the membership product instead
                    const bool fin = __builtin_isfinite(b[tj]);
                    bf[tj] = fin ? 0.0 : 1.0;
                    b[tj] = fin ? b[tj] : 0.0;
                }
            }
            acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b[0], acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b[1], acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b[0], acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b[1], acc[1][1], 0, 0, 0);
            if (FLAG) {
                const double f0 = m0[k0], f1 = m1[k0];
                accf[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0, bf[0], accf[0][0], 0, 0, 0);
                accf[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0, bf[1], accf[0][1], 0, 0, 0);
                accf[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(f1, bf[0], accf[1][0], 0, 0, 0);
                accf[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(f1, bf[1], accf[1][1], 0, 0, 0);
            }
            xk += 4 * a.slot_stride;
        }
        if (FLAG) {
            // an output that one of the event's non-finite members reaches is NaN, as the
            // reference's sum over the event's own sources gives
            for (int ti = 0; ti < 2; ti++)
                for (int tj = 0; tj < 2; tj++)
                    for (int r = 0; r < 4; r++)
                        if (accf[ti][tj][r] != 0.0) acc[ti][tj][r] = __builtin_nan("");
        }
        if (MODE == 0) {
            for (int ti = 0; ti < 2; ti++)
                for (int r = 0; r < 4; r++) {
                    const int e = e_base + ti * 16 + lk + 4 * r;
                    if (e >= a.E) continue;
                    for (int tj = 0; tj < 2; tj++)
                        if (cok[tj])
                            a.out[(long long)e * N + caddr[tj]] = acc[ti][tj][r] * scale[ti][r] + offs[ti][tj][r];
                }
        } else {
            for (int ti = 0; ti < 2; ti++)
                for (int tj = 0; tj < 2; tj++)
                    for (int r = 0; r < 4; r++)
                        if (s < nval[ti][r]) {
                            const double v = acc[ti][tj][r] * scale[ti][r] + offs[ti][tj][r];
                            mx[ti][tj][r] = v > mx[ti][tj][r] ? v : mx[ti][tj][r];
                            if (FLAG && v != v) nan_seen[ti][tj][r] = true;   // a maximum over NaN is NaN
                        }
        }
    }
    if (MODE == 1) {
        for (int ti = 0; ti < 2; ti++)
            for (int r = 0; r < 4; r++) {
                const int e = e_base + ti * 16 + lk + 4 * r;
                if (e >= a.E) continue;
                for (int tj = 0; tj < 2; tj++) {
                    if (!cok[tj]) continue;
                    double *o = a.out + (long long)e * a.ng + caddr[tj];
                    if (FLAG && nan_seen[ti][tj][r])
                        // NaN stays: atomic_max_f64 never replaces it (NaN < v is false)
                        atomicExch(reinterpret_cast<unsigned long long *>(o),
                                   (unsigned long long)__double_as_longlong(__builtin_nan("")));
                    else if (mx[ti][tj][r] > -__builtin_huge_val())
                        atomic_max_f64(o, mx[ti][tj][r], __hip_atomic_load(o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                }
            }
    }
}

// The same events from lists of their sources. A hazard event ruptures a patch of a source
// zone, so a dense product over all sources spends most of its work on zero weights; here a
// workgroup stages one tile of columns of every source in LDS (2 L columns: 512 sources of
// 32 columns are 128 KB, one workgroup per CU) and every event sums its own sources' rows
// from there, L lanes per event with two columns each, so a wavefront takes 64 / L events.
// MODE 0: the tile is 2 L consecutive columns. MODE 1: L gauges of two samples, whose
// maximum the lane takes before it meets the event's maximum in memory. What bounds it: LDS
// reads (256 B per event, source and tile) and, where events have few sources, the chain of
// an event's record, list and maximum, which are asked for one event ahead (4096 events of
// 38 in 512 sources: 1.7 -> 1.44 ms with that).
constexpr int kListThreads = 1024;

template <int MODE, int L, bool WEIGHTS>
__global__ __launch_bounds__(kListThreads) void superpose_lists_kernel(SupArgs a)
{
    extern __shared__ __align__(16) double tile[];   // [nsrc + 1][2 L]; the last row zero
    constexpr int C = 2 * L;
    const long long N = (long long)a.gmax * 3 * a.ng;
    const int t = threadIdx.x, li = t % L;
    // MODE 0: first column; MODE 1: first gauge and first sample
    const long long c0 = (long long)blockIdx.x * C;
    const int gtiles = (a.ng + L - 1) / L;
    const int g0 = MODE == 1 ? (int)(blockIdx.x % gtiles) * L : 0, s0 = MODE == 1 ? (int)(blockIdx.x / gtiles) * 2 : 0;
    {
        const int c = t % C, half = c / L, gg = g0 + c % L;
        const bool ok = MODE == 0 ? c0 + c < N : gg < a.ng && s0 + half < a.s_max;
        const long long src = MODE == 0 ? c0 + c : (long long)(s0 + half) * 3 * a.ng + gg;
        const double sub = MODE == 1 || (src / a.ng) % 3 == 0 ? a.msl : 0.0;   // stage - msl is linear
        const int at = MODE == 0 ? c : 2 * (c % L) + half;
        for (int k = t / C; k <= a.nsrc; k += kListThreads / C) {
            double x = ok && k < a.nsrc ? a.X[(long long)k * a.slot_stride + src] - sub : 0.0;
            if (a.flagged && !__builtin_isfinite(x)) x = __builtin_nan("");
            tile[k * C + at] = x;
        }
    }
    __syncthreads();
    const double2 *rows = reinterpret_cast<const double2 *>(tile) + li;
    const int step = (int)gridDim.y * (kListThreads / L);
    int q = (int)blockIdx.y * (kListThreads / L) + t / L;
    if (q >= a.E) return;
    // two list entries of four sources ahead (the lists end in two spare ones), and the next
    // event's record and first entries beside this one's sum
    const ushort4 *ls = reinterpret_cast<const ushort4 *>(a.lists);
    SupList ev = a.recs[q];
    ushort4 n0 = ls[ev.begin], n1 = ls[ev.begin + 1];
    for (; q < a.E; q += step) {
        const SupList cur = ev;
        const int b = cur.begin, end = cur.begin + cur.n;
        if (q + step < a.E) ev = a.recs[q + step];
        double acc0 = 0.0, acc1 = 0.0;
        // the event's maximum so far, asked for early: no atomic where the value is no larger
        double *o = a.out;
        double seen = 0.0;
        if (MODE == 1) {
            o += (long long)cur.event * a.ng + min(g0 + li, a.ng - 1);
            seen = __hip_atomic_load(o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        for (int k = b; k < end; k++) {
            const ushort4 c = n0;
            n0 = n1;
            n1 = ls[k + 2];
            const double2 x0 = rows[c.x * L], x1 = rows[c.y * L], x2 = rows[c.z * L], x3 = rows[c.w * L];
            if (WEIGHTS) {
                const double *w = a.list_w + 4LL * k;
                acc0 = __builtin_fma(w[0], x0.x, acc0); acc1 = __builtin_fma(w[0], x0.y, acc1);
                acc0 = __builtin_fma(w[1], x1.x, acc0); acc1 = __builtin_fma(w[1], x1.y, acc1);
                acc0 = __builtin_fma(w[2], x2.x, acc0); acc1 = __builtin_fma(w[2], x2.y, acc1);
                acc0 = __builtin_fma(w[3], x3.x, acc0); acc1 = __builtin_fma(w[3], x3.y, acc1);
            } else {
                acc0 += x0.x; acc1 += x0.y;
                acc0 += x1.x; acc1 += x1.y;
                acc0 += x2.x; acc1 += x2.y;
                acc0 += x3.x; acc1 += x3.y;
            }
        }
        n0 = ls[ev.begin];
        n1 = ls[ev.begin + 1];
        const double scale = cur.scale;
        const int e = cur.event;
        if (MODE == 0) {
            const long long c = c0 + 2 * li;
            const double o0 = (c / a.ng) % 3 == 0 ? a.msl : 0.0, o1 = ((c + 1) / a.ng) % 3 == 0 ? a.msl : 0.0;
            if (c < N) a.out[(long long)e * N + c] = acc0 * scale + o0;
            if (c + 1 < N) a.out[(long long)e * N + c + 1] = acc1 * scale + o1;
        } else if (g0 + li < a.ng) {
            const int nv = min(cur.nvalid, a.s_max);
            const double v0 = acc0 * scale + a.msl, v1 = acc1 * scale + a.msl;
            double mx = -__builtin_huge_val();
            if (s0 < nv && v0 > mx) mx = v0;
            if (s0 + 1 < nv && v1 > mx) mx = v1;
            if (a.flagged && ((s0 < nv && v0 != v0) || (s0 + 1 < nv && v1 != v1)))
                // NaN stays: atomic_max_f64 never replaces it (NaN < v is false)
                atomicExch(reinterpret_cast<unsigned long long *>(o),
                           (unsigned long long)__double_as_longlong(__builtin_nan("")));
            else if (mx > seen)
                atomic_max_f64(o, mx, seen);
        }
    }
}

__global__ void nonfinite_slots_kernel(const double *__restrict__ X, long long slot_stride, int *flags)
{
    const int slot = blockIdx.y;
    const double *x = X + (long long)slot * slot_stride;
    bool bad = false;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < slot_stride;
         i += (long long)gridDim.x * blockDim.x)
        bad |= !__builtin_isfinite(x[i]);
    if (bad) flags[slot] = 1;   // every writer stores the same value
}

__global__ void fill_kernel(double *p, long long n, double v)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace

int superpose_event_tile() { return kTE; }

hipError_t launch_superpose(const SupArgs &a, int mode, hipStream_t s)
{
    if (a.Kpad % 4 || a.Kpad < a.nsrc || a.E <= 0 || a.ng <= 0 || a.gmax <= 0) return hipErrorInvalidValue;
    const int ety = (a.E + kTE - 1) / kTE;
    if (mode == 0) {
        const long long N = (long long)a.gmax * 3 * a.ng;
        if (N >= (1LL << 31)) return hipErrorInvalidValue;
        if (a.M)
            hipLaunchKernelGGL((superpose_kernel<0, true>), dim3((unsigned)((N + kTN - 1) / kTN), ety), dim3(256), 0,
                               s, a);
        else
            hipLaunchKernelGGL((superpose_kernel<0, false>), dim3((unsigned)((N + kTN - 1) / kTN), ety), dim3(256), 0,
                               s, a);
    } else {
        if (a.s_chunk < 1 || a.s_max < 1 || a.s_max > a.gmax) return hipErrorInvalidValue;
        const long long n = (long long)a.E * a.ng;
        hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a.out, n,
                           -__builtin_huge_val());
        const int nz = (a.s_max + a.s_chunk - 1) / a.s_chunk;
        if (a.M)
            hipLaunchKernelGGL((superpose_kernel<1, true>), dim3((a.ng + kTN - 1) / kTN, ety, nz), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((superpose_kernel<1, false>), dim3((a.ng + kTN - 1) / kTN, ety, nz), dim3(256), 0, s,
                               a);
    }
    return hipGetLastError();
}

template <int MODE, int L, bool WEIGHTS>
static hipError_t launch_lists(const SupArgs &a, hipStream_t s)
{
    const size_t lds = (size_t)(a.nsrc + 1) * 2 * L * sizeof(double);
    const void *k = (const void *)superpose_lists_kernel<MODE, L, WEIGHTS>;
    hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const long long N = (long long)a.gmax * 3 * a.ng;
    const long long tiles = MODE == 0 ? (N + 2 * L - 1) / (2 * L)
                                      : (long long)((a.ng + L - 1) / L) * ((a.s_max + 1) / 2);
    // a few rounds of workgroups: events are split where the tiles are few
    const int per = kListThreads / L;
    const long long split = std::min<long long>((a.E + per - 1) / per, std::max<long long>(1, 1024 / tiles));
    hipLaunchKernelGGL((superpose_lists_kernel<MODE, L, WEIGHTS>), dim3((unsigned)tiles, (unsigned)split),
                       dim3(kListThreads), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_superpose_lists(const SupArgs &a, int mode, hipStream_t s)
{
    const int L = list_lanes(a.nsrc);
    const long long N = (long long)a.gmax * 3 * a.ng;
    if (!L || a.E <= 0 || a.ng <= 0 || a.gmax <= 0 || a.nsrc < 1 || N >= (1LL << 31) || !a.recs || !a.lists)
        return hipErrorInvalidValue;
    if (mode == 0) {
        if (L == 16) return a.list_w ? launch_lists<0, 16, true>(a, s) : launch_lists<0, 16, false>(a, s);
        return a.list_w ? launch_lists<0, 8, true>(a, s) : launch_lists<0, 8, false>(a, s);
    }
    if (a.s_max < 1 || a.s_max > a.gmax) return hipErrorInvalidValue;
    const long long n = (long long)a.E * a.ng;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a.out, n, -__builtin_huge_val());
    if (L == 16) return a.list_w ? launch_lists<1, 16, true>(a, s) : launch_lists<1, 16, false>(a, s);
    return a.list_w ? launch_lists<1, 8, true>(a, s) : launch_lists<1, 8, false>(a, s);
}

hipError_t launch_nonfinite_slots(const double *X, int nsrc, long long slot_stride, int *flags, hipStream_t s)
{
    if (nsrc < 1 || nsrc > 65535 || slot_stride < 1) return hipErrorInvalidValue;
    const long long per = (slot_stride + 255) / 256;
    const unsigned gx = (unsigned)std::min<long long>(per, 64);
    hipLaunchKernelGGL(nonfinite_slots_kernel, dim3(gx, nsrc), dim3(256), 0, s, X, slot_stride, flags);
    return hipGetLastError();
}

}  // namespace swh
