// remc_analysis.hip -- device reductions over the live replica conformations.
//
//   k_drms             distance RMS of every replica of a system against a
//                      reference conformation, over bead pairs of different
//                      non-crowder bodies ("post processor/pdbgensrc/
//                      drms.cpp:7-58"): one workgroup per (64-row x column
//                      tile, four replicas); FP32 distances, FP64 sums, tiles
//                      added in fixed order.
//   k_centre_hist      histogram of body-centre distances (minimum image,
//                      FP64) by body-type pair over every replica of a system
//                      ("post processor/gr.py:93-140"): every unordered pair
//                      once, one LDS histogram per workgroup;
//   k_hist_out         their sum, as counts or as g(r).
#include <algorithm>

#include "remc_internal.h"

namespace remc {

constexpr int DRMS_ROWS = 64;  // row beads of a unit, one per lane
constexpr int DRMS_WAVES = 4;  // waves, each on a quarter of the unit's columns
constexpr int DRMS_REPS = 4;   // replicas of a unit: the reference distance of a pair is formed once for them
constexpr int DRMS_COLS = 256; // most columns of a unit

// FP32 Euclidean distance: the fused sum of squares is written out, so that
// the conformation's and the reference's distance of a pair round alike
// wherever they are formed (a conformation equal to the reference gives 0).
__device__ __forceinline__ float plain_dist(float dx, float dy, float dz)
{
    return __fsqrt_rn(__builtin_fmaf(dz, dz, __builtin_fmaf(dx, dx, dy * dy)));
}

// Unit (row tile, column tile, replica group) = blockIdx (x / nct, x % nct, y);
// partials[(replica k) * units + x].  Bound by FP32 VALU (the correctly rounded
// square roots); small units keep every SIMD in several waves, where one
// workgroup per 256-row tile walked all its column tiles (the first one 43
// times the last one's work at 11,000 beads).
// 32 x 1300 beads: 195 -> 21 us.
__global__ __launch_bounds__(64 * DRMS_WAVES) void k_drms(KParams p, int sys_id, const float *rx, const float *ry,
                                                          const float *rz, double *partials, int n_rep, int cols, int nct)
{
    __shared__ float4 s_ref[DRMS_COLS]; // reference position; w: body (-1: crowder), as bits
    __shared__ float s_p[DRMS_REPS][3][DRMS_COLS];
    __shared__ double s_red[DRMS_WAVES][DRMS_REPS];
    const DevSys S = p.sys[sys_id];
    const int N = S.n_beads;
    const int x = blockIdx.x, i0 = (x / nct) * DRMS_ROWS, j0 = (x % nct) * cols;
    const int k0 = blockIdx.y * DRMS_REPS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (j0 + cols <= i0 + 1) { // no pair j > i
        if (tid < DRMS_REPS && k0 + tid < n_rep) partials[(size_t)(k0 + tid) * gridDim.x + x] = 0.0;
        return;
    }
    const int *body = p.body + S.bead_off;
    const int *crow = p.bcrow + S.body_off;
    // a replica past the last repeats it (its sum is dropped)
    int off[DRMS_REPS];
#pragma unroll
    for (int q = 0; q < DRMS_REPS; ++q) off[q] = p.rep[S.rep_first + min(k0 + q, n_rep - 1)].bead_off;
    for (int t = tid; t < cols; t += 64 * DRMS_WAVES) {
        const int j = j0 + t;
        int bj = -1;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < N) {
            bj = body[j];
            if (crow[bj]) bj = -1;
            v = make_float4(rx[j], ry[j], rz[j], 0.f);
#pragma unroll
            for (int q = 0; q < DRMS_REPS; ++q) {
                s_p[q][0][t] = p.px[off[q] + j];
                s_p[q][1][t] = p.py[off[q] + j];
                s_p[q][2][t] = p.pz[off[q] + j];
            }
        }
        v.w = __int_as_float(bj);
        s_ref[t] = v;
    }
    const int i = i0 + lane;
    int bi = -1;
    float ax = 0.f, ay = 0.f, az = 0.f, xi[DRMS_REPS] = {}, yi[DRMS_REPS] = {}, zi[DRMS_REPS] = {};
    if (i < N) {
        bi = body[i];
        if (crow[bi]) bi = -1;
        ax = rx[i];
        ay = ry[i];
        az = rz[i];
#pragma unroll
        for (int q = 0; q < DRMS_REPS; ++q) {
            xi[q] = p.px[off[q] + i];
            yi[q] = p.py[off[q] + i];
            zi[q] = p.pz[off[q] + i];
        }
    }
    __syncthreads();
    double acc[DRMS_REPS] = {};
    const int per = cols / DRMS_WAVES, t1 = (wave + 1) * per;
    for (int t = wave * per; t < t1; ++t) {
        const float4 v = s_ref[t];
        const int bj = __float_as_int(v.w);
        if (!(bi >= 0 && bj >= 0 && bj != bi && j0 + t > i)) continue;
        const float e = plain_dist(ax - v.x, ay - v.y, az - v.z);
#pragma unroll
        for (int q = 0; q < DRMS_REPS; ++q) {
            const float d = plain_dist(xi[q] - s_p[q][0][t], yi[q] - s_p[q][1][t], zi[q] - s_p[q][2][t]);
            acc[q] += (double)fabsf(__fsub_rn(d, e)); // |float - float| as the reference's abs of magnitudes
        }
    }
#pragma unroll
    for (int q = 0; q < DRMS_REPS; ++q) {
        for (int o = 32; o > 0; o >>= 1) acc[q] += __shfl_xor(acc[q], o, 64);
        if (lane == 0) s_red[wave][q] = acc[q];
    }
    __syncthreads();
    if (tid < DRMS_REPS && k0 + tid < n_rep) {
        double t = 0.0;
        for (int w = 0; w < DRMS_WAVES; ++w) t += s_red[w][tid];
        partials[(size_t)(k0 + tid) * gridDim.x + x] = t;
    }
}

// one wave per replica: lane l adds units l, l + 64, ..., then a fixed butterfly
__global__ __launch_bounds__(64) void k_drms_sum(const double *partials, int units, double inv_pairs, double *out,
                                                 Signal sig)
{
    const int k = blockIdx.x, lane = threadIdx.x;
    double t = 0.0;
    for (int i = lane; i < units; i += 64) t += partials[(size_t)k * units + i];
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane == 0) host_store(out + k, t * inv_pairs);
    signal_done(sig);
}

// Columns per unit: 64 until the launch holds enough units for every SIMD to
// have several waves at 256 (four times fewer stagings and partials a pair).
static int drms_cols(int n_beads, int n_rep)
{
    const long long rows = (n_beads + DRMS_ROWS - 1) / DRMS_ROWS, groups = (n_rep + DRMS_REPS - 1) / DRMS_REPS;
    return rows * ((n_beads + DRMS_COLS - 1) / DRMS_COLS) * groups >= 4096 ? DRMS_COLS : 64;
}

size_t drms_units(int n_beads, int n_rep)
{
    const int cols = drms_cols(n_beads, n_rep);
    return (size_t)((n_beads + DRMS_ROWS - 1) / DRMS_ROWS) * ((n_beads + cols - 1) / cols);
}

hipError_t launch_drms(const KParams &p, int sys_id, int n_beads, int n_rep, const float *rx, const float *ry,
                       const float *rz, double *partials, double inv_pairs, double *out, const Signal &sig, hipStream_t s)
{
    if (n_rep <= 0 || n_beads <= 0) return hipSuccess;
    const int cols = drms_cols(n_beads, n_rep), nct = (n_beads + cols - 1) / cols;
    const int units = (int)drms_units(n_beads, n_rep);
    hipLaunchKernelGGL(k_drms, dim3(units, (n_rep + DRMS_REPS - 1) / DRMS_REPS), dim3(64 * DRMS_WAVES), 0, s, p, sys_id,
                       rx, ry, rz, partials, n_rep, cols, nct);
    hipLaunchKernelGGL(k_drms_sum, dim3(n_rep), dim3(64), 0, s, partials, units, inv_pairs, out, sig);
    return hipGetLastError();
}

constexpr int HIST_TILE = 64;  // bodies per side of a unit: lanes hold the rows
constexpr int HIST_WAVES = 4;  // waves, each on a quarter of the unit's columns

// x / d to the nearest double rounded down, and to the nearest whole number
// (halves away from zero) as round(x / d) gives it, from the product with inv
// = 1/d: the product and the quotient differ by a few units in the last
// place, so the division is only formed where the product lies that near to a
// value at which the result changes.
__device__ __forceinline__ double floor_quotient(double x, double d, double inv)
{
    const double q = x * inv;
    return fabs(q - rint(q)) > 1e-14 * fabs(q) ? floor(q) : floor(__ddiv_rn(x, d)); // (an infinite q divides)
}

__device__ __forceinline__ double round_quotient(double x, double d, double inv)
{
    const double t = fabs(x) * inv + 0.5;
    return fabs(t - rint(t)) > 1e-14 * t ? copysign(floor(t), x) : round(__ddiv_rn(x, d));
}

// part[g * nh + (ti * n_types + tj) * nbin + bin] of workgroup g, for ti <= tj:
// a pair of bodies of the same type counts twice (once from each side), a pair
// of different types once (gr.py's loops over typeI <= typeJ and over both
// chains).  A body's point is its centre, or with `site` the position of its
// bead site[m] (gr.py takes the residue nearest each chain's centroid).
//
// Workgroup g takes a contiguous share of the n_rep x T (T + 1) / 2 units
// (replica, row tile a, column tile b >= a); a wave reads its 16 columns into
// lanes and broadcasts them one by one.  Latency bound at the sizes that
// occur, so the work is spread over the device and the divisions of the
// minimum image and of the bin (four per pair in FP64) become products.
// 32 x 310 bodies, 480 bins: 127 -> 13 us, and 5 for k_hist_out.
__global__ __launch_bounds__(64 * HIST_WAVES) void k_centre_hist(KParams p, int sys_id, int n_rep, const int *btype,
                                                                 const int *site, int n_types, int nbin, double lo,
                                                                 double dr, unsigned int *part)
{
    extern __shared__ unsigned int s_hist[];
    const DevSys S = p.sys[sys_id];
    const int M = S.n_bodies, T = (M + HIST_TILE - 1) / HIST_TILE;
    const int nh = n_types * n_types * nbin;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int t = tid; t < nh; t += 64 * HIST_WAVES) s_hist[t] = 0u;
    __syncthreads();
    const double L = (double)S.box, inv_L = L > 0.0 ? 1.0 / L : 0.0, inv_dr = 1.0 / dr;
    const long long per_rep = (long long)T * (T + 1) / 2, all = per_rep * n_rep;
    long long u = all * blockIdx.x / gridDim.x;
    const long long u1 = all * (blockIdx.x + 1) / gridDim.x;
    int k = (int)(u / per_rep), a = 0;
    long long left = u % per_rep;
    while (left >= T - a) left -= T - a++;
    int b = a + (int)left;
    for (; u < u1; ++u) {
        const DevRep R = p.rep[S.rep_first + k];
        const float *fx = site ? p.px + R.bead_off : p.cx + R.body_off;
        const float *fy = site ? p.py + R.bead_off : p.cy + R.body_off;
        const float *fz = site ? p.pz + R.bead_off : p.cz + R.body_off;
        const int i = a * HIST_TILE + lane;
        int ti = -1;
        double xi = 0.0, yi = 0.0, zi = 0.0;
        if (i < M) {
            ti = btype[i];
            if (ti >= 0) { // a body left out has no site
                const int w = site ? site[i] : i;
                xi = fx[w];
                yi = fy[w];
                zi = fz[w];
            }
        }
        constexpr int PER = HIST_TILE / HIST_WAVES;
        const int jl = b * HIST_TILE + wave * PER + (lane & (PER - 1));
        int tl = -1;
        float xl = 0.f, yl = 0.f, zl = 0.f;
        if (jl < M) {
            tl = btype[jl];
            if (tl >= 0) {
                const int w = site ? site[jl] : jl;
                xl = fx[w];
                yl = fy[w];
                zl = fz[w];
            }
        }
#pragma unroll 2
        for (int t = 0; t < PER; ++t) {
            const int j = b * HIST_TILE + wave * PER + t;
            const int tj = __builtin_amdgcn_readlane(tl, t);
            if (tj < 0) continue;
            const float xj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xl), t));
            const float yj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(yl), t));
            const float zj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(zl), t));
            if (ti < 0 || j <= i) continue;
            double dx = __dsub_rn(xi, (double)xj), dy = __dsub_rn(yi, (double)yj), dz = __dsub_rn(zi, (double)zj);
            if (L > 0.0) {
                dx = __dsub_rn(dx, __dmul_rn(L, round_quotient(dx, L, inv_L)));
                dy = __dsub_rn(dy, __dmul_rn(L, round_quotient(dy, L, inv_L)));
                dz = __dsub_rn(dz, __dmul_rn(L, round_quotient(dz, L, inv_L)));
            }
            const double r = __dsqrt_rn(__dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz)));
            const double f = floor_quotient(__dsub_rn(r, lo), dr, inv_dr);
            if (!(f >= 0.0 && f < (double)nbin)) continue;
            atomicAdd(&s_hist[(min(ti, tj) * n_types + max(ti, tj)) * nbin + (int)f], ti == tj ? 2u : 1u);
        }
        if (++b == T) {
            if (++a == T) {
                a = 0;
                ++k;
            }
            b = a;
        }
    }
    __syncthreads();
    for (int t = tid; t < nh; t += 64 * HIST_WAVES) part[(size_t)blockIdx.x * nh + t] = s_hist[t];
}

// The workgroups' histograms added: as counts, or (gr not null) as
// g = counts / (frames 4 pi r^2 dr n_ti n_tj / V), r the bin centre
// (gr.py:140-155).  16 bins per workgroup, 64 groups of threads on a share of
// the histograms each: the histograms come from other XCDs' caches, so the
// loads of a share are kept few and in flight together.
constexpr int HOUT_BINS = 16, HOUT_GROUPS = 64;
__global__ __launch_bounds__(HOUT_BINS * HOUT_GROUPS) void k_hist_out(const unsigned int *part, int n_part,
                                                                      const int *type_count, int n_types, int nbin,
                                                                      double lo, double dr, double frames_over_volume,
                                                                      unsigned long long *counts, double *gr, Signal sig)
{
    __shared__ unsigned long long s_sum[HOUT_GROUPS][HOUT_BINS];
    const int nh = n_types * n_types * nbin;
    const int bin = threadIdx.x % HOUT_BINS, group = threadIdx.x / HOUT_BINS;
    const int t = blockIdx.x * HOUT_BINS + bin;
    unsigned long long c = 0ull;
    if (t < nh)
#pragma unroll 8
        for (int g = group; g < n_part; g += HOUT_GROUPS) c += part[(size_t)g * nh + t];
    s_sum[group][bin] = c;
    __syncthreads();
    if (group == 0 && t < nh) {
        for (int w = 1; w < HOUT_GROUPS; ++w) c += s_sum[w][bin];
        const int b = t % nbin, pair = t / nbin, ti = pair / n_types, tj = pair % n_types;
        if (!gr) {
            host_store(counts + t, c);
        } else if (ti > tj) {
            host_store(gr + t, 0.0);
        } else {
            const double r = lo + (0.5 + (double)b) * dr;
            const double four_pi = 12.566370614359172953850573533118;
            const double norm = frames_over_volume * four_pi * r * r * dr * (double)type_count[ti] * (double)type_count[tj];
            host_store(gr + t, norm > 0.0 ? (double)c / norm : 0.0);
        }
    }
    signal_done(sig);
}

// Workgroups of the histogram: one a unit up to four a CU; fewer where their
// histograms would hold more than 2^21 bins, more where one's 32-bit counts
// could overflow (a unit adds at most 2 x 64 x 64).
int hist_workgroups(int n_bodies, int n_rep, int nh)
{
    const long long T = (n_bodies + HIST_TILE - 1) / HIST_TILE, units = T * (T + 1) / 2 * n_rep;
    const long long cap = std::max<long long>(64, std::min<long long>(1024, (1 << 21) / nh));
    return (int)std::min(units, std::max(cap, (units >> 18) + 1));
}

hipError_t launch_centre_hist(const KParams &p, int sys_id, int n_bodies, int n_rep, const int *btype, const int *site,
                              int n_types, int nbin, double lo, double dr, unsigned int *part, const int *type_count,
                              double frames_over_volume, unsigned long long *counts, double *gr, const Signal &sig, hipStream_t s)
{
    if (n_rep <= 0 || n_bodies <= 0) return hipSuccess;
    const int nh = n_types * n_types * nbin, n_part = hist_workgroups(n_bodies, n_rep, nh);
    hipLaunchKernelGGL(k_centre_hist, dim3(n_part), dim3(64 * HIST_WAVES), sizeof(unsigned int) * (size_t)nh, s, p, sys_id,
                       n_rep, btype, site, n_types, nbin, lo, dr, part);
    hipLaunchKernelGGL(k_hist_out, dim3((nh + HOUT_BINS - 1) / HOUT_BINS), dim3(HOUT_BINS * HOUT_GROUPS), 0, s, part, n_part,
                       type_count, n_types, nbin, lo, dr, frames_over_volume, counts, gr, sig);
    return hipGetLastError();
}

} // namespace remc
