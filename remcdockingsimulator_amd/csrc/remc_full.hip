// remc_full.hip -- kernels over all pairs of a replica.
//
//   k_energy_full      batched full energy, every replica in one launch: each
//                      unordered pair of 64-bead tiles once (half-window
//                      schedule), FP32 pair terms, FP64 sums; k_sum_partials
//                      adds the units in fixed order.
//   k_adjoint_rows/_bodies  gradient of the energy: per-body force and torque,
//                      d/d(lambda, e0, xi).
//
// Both give a workgroup 64 row beads (one per lane, the same rows in each of
// its four waves) and walk partner columns in groups of 16 beads, one group per
// wave at a time.  They are bound by VALU issue (4 cycles an instruction of a
// wave, 8 a transcendental one), so a group is classified once for the whole
// wave from a summary that is made ahead, columns come in by scalar loads
// (they are uniform, and cost the vector pipes nothing; a broadcast read from
// LDS returns 64 lanes' worth of data a column), and the work per pair is cut
// to what the class needs:
//   - the minimum image.  d - L rint(d/L) costs four instructions an axis in
//     floating point.  In boxes of up to FIX_BOX_MAX k_fix writes every
//     coordinate as a 32-bit fraction of the box: the difference of two wraps to
//     the nearest image by itself, in one subtraction and one conversion.
//     Contact distances are in that unit, with the constants scaled to it
//     (sigma_ij^2 as a sum of two floats: rounded to one, its error would be the
//     same in every pair and add up).  Larger boxes and systems without one take
//     float differences in Angstrom (CoordForm).  Crowder pairs
//     keep the float form, which decides what lies inside their cutoff.
//   - crowder pairs end at 15 A.  The crowder columns of a chain's rows are
//     screened by their distance from the rows' groups against the groups'
//     extent (triangle inequality), 16 columns x 4 row groups in one step, and a
//     chain's group against crowder rows by the group's extent; most of them go.
//   - the repulsive flip and the 1e30 cap can only act where x6 > 1/2: they
//     sit behind one wave-wide test.  Debye-Hueckel is formed for charged
//     columns only (a scalar branch).
// Contact pairs of rows and columns that share bodies or kinds, or lie in the
// diagonal tile, are formed by the same code with a mask per pair.
#include <algorithm>
#include <type_traits>

#include "remc_internal.h"
#include "remc_math.h"
#include "remc_pair.h"

namespace remc {

constexpr int ROWS = 64;                // row beads of a workgroup (a tile)
constexpr int WAVES = 4;                // waves of a workgroup
constexpr int COLS = 64 * WAVES;        // threads of a workgroup
constexpr int TSTRIDE = REMC_NTYPES + 1; // row stride of the type tables in LDS: 21 entries keep rows on different banks

// How a system's contact distances are formed.  A fraction of a box L is rounded
// to L 2^-32, so a difference of two is off by up to that much, where the
// difference of two near floats is exact: at 1024 A it is 2^-22 A, what a
// difference of 4-8 A (a contact's) may be off by when rounded to 24 bits, and it
// grows with the box.  Root mean square error of (sigma/r)^6, pairs 4.5-8 A apart
// anywhere in the box (emulated, reciprocals off by half a unit): 2.2e-7 at
// 150 A, 2.3e-7 at 600, 2.5e-7 at 1000, 5.1e-7 at 5000, 9.5e-5 at 1e6 A; float
// differences 1.8e-7 in any box, and 3.0e-7 with a squared reciprocal root, as
// the general form of a term has (pair_lj_dh).  Fractions take two instructions
// less an axis: 64 x 11000 beads 1.74 ms an energy launch and 5.04 an adjoint's,
// 1.84 and 5.25 with float differences; 32 x 1300 beads 43.4 and 83 us with both.
enum CoordForm {
    FRACTION, // fractions of the box
    IMAGE,    // float differences, nearest image
    FLAT      // float differences, no box
};
template <CoordForm F>
using Form = std::integral_constant<CoordForm, F>;

// A replica's beads and groups for reads at wave-uniform indices: through the
// constant address space they become scalar loads.  Nothing writes these arrays
// while the kernels run.
template <typename T>
using Uniform = const __attribute__((address_space(4))) T *;
struct Beads {
    Uniform<float> x, y, z, q, s;
    Uniform<int> tc, body, fx, fy, fz; // fx..: coordinates as fractions of the box (k_fix)
    Uniform<int> g;                    // per group: first body, last body, kinds | beads << 8, mask of the charged beads
    Uniform<float> c;                  // per group: middle of its coordinates' range and half its diagonal
};

// Full min over / max over each row of 16 lanes.
template <bool MAX>
__device__ __forceinline__ float row16(float v)
{
#define REMC_ROW_STEP(ctrl)                                                                                    \
    {                                                                                                          \
        const float o = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true)); \
        v = MAX ? fmaxf(v, o) : fminf(v, o);                                                                   \
    }
    REMC_ROW_STEP(0x128) // row_ror:8
    REMC_ROW_STEP(0x124)
    REMC_ROW_STEP(0x122)
    REMC_ROW_STEP(0x121)
#undef REMC_ROW_STEP
    return v;
}

// A lane's row bead and what the wave knows of its 64 rows.  Lanes past the
// last bead (not on) repeat it, so that every lane takes part in the wave's
// votes; their sums are dropped.
struct Row {
    float x, y, z;
    int i, body, type;
    bool on, crow;
    int kinds, b0, b1; // kinds and body range of the rows (uniform)
    int g0, gn;        // their first group and its number of groups (uniform)
    float size;        // their largest |x| + |y| + |z| (uniform, screen_limit)
};

__device__ __forceinline__ Row load_row(int tile, int N, const float *gx, const float *gy, const float *gz, const int *tcs,
                                        const int *bodies)
{
    Row r;
    const int lane = threadIdx.x & 63;
    r.i = tile * ROWS + lane;
    r.on = r.i < N;
    const int i = r.on ? r.i : N - 1;
    r.x = gx[i];
    r.y = gy[i];
    r.z = gz[i];
    const int tc = tcs[i];
    r.type = tc & 0xff;
    r.crow = (tc >> 8) != 0;
    r.body = bodies[i];
    const unsigned long long cm = __ballot(r.crow);
    r.kinds = (~cm ? GROUP_CHAIN : 0) | (cm ? GROUP_CROWDER : 0);
    r.b0 = __builtin_amdgcn_readlane(r.body, 0);
    r.b1 = __builtin_amdgcn_readlane(r.body, 63);
    r.g0 = tile * (ROWS / GROUP);
    r.gn = min(ROWS / GROUP, full_groups(N) - r.g0);
    const int s = __float_as_int(row16<true>(fabsf(r.x) + fabsf(r.y) + fabsf(r.z)));
    const float s0 = __int_as_float(__builtin_amdgcn_readlane(s, 0)), s1 = __int_as_float(__builtin_amdgcn_readlane(s, 16)),
                s2 = __int_as_float(__builtin_amdgcn_readlane(s, 32)), s3 = __int_as_float(__builtin_amdgcn_readlane(s, 48));
    r.size = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fmaxf(fmaxf(s0, s1), fmaxf(s2, s3)))));
    return r;
}

// The lane's row as fractions of the box (FRACTION).
struct RowFix {
    int x, y, z;
};
__device__ __forceinline__ RowFix load_row_fix(const Row &r, const int *fx, const int *fy, const int *fz, int N)
{
    const int i = r.on ? r.i : N - 1;
    return {fx[i], fy[i], fz[i]};
}

// A column's bead as the contact pairs read it (uniform): coordinates as
// fractions of the box (FRACTION) or in Angstrom.
struct Column {
    int fx, fy, fz, tc;
    float x, y, z, q, s;
};
template <bool TAB, CoordForm FORM, int N>
__device__ __forceinline__ void load_columns(const Beads &B, int j, Column *c)
{
    const auto fx = B.fx + j, fy = B.fy + j, fz = B.fz + j, tc = B.tc + j;
    const auto x = B.x + j, y = B.y + j, z = B.z + j, q = B.q + j, s = B.s + j;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if (FORM == FRACTION) {
            c[k].fx = fx[k];
            c[k].fy = fy[k];
            c[k].fz = fz[k];
        } else {
            c[k].x = x[k];
            c[k].y = y[k];
            c[k].z = z[k];
        }
        c[k].tc = tc[k];
        c[k].q = q[k];
        if (!TAB) c[k].s = s[k];
    }
}

// Column minus the lane's row, nearest image.
template <CoordForm FORM>
__device__ __forceinline__ void separation(const Column &c, const Row &r, const RowFix &f, const DevSys &S, float &dx,
                                           float &dy, float &dz)
{
    if (FORM == FRACTION) {
        dx = (float)(int)((unsigned)c.fx - (unsigned)f.x);
        dy = (float)(int)((unsigned)c.fy - (unsigned)f.y);
        dz = (float)(int)((unsigned)c.fz - (unsigned)f.z);
    } else {
        dx = c.x - r.x;
        dy = c.y - r.y;
        dz = c.z - r.z;
        if (FORM == IMAGE) {
            dx = min_image(dx, S.box, S.inv_box);
            dy = min_image(dy, S.box, S.inv_box);
            dz = min_image(dz, S.box, S.inv_box);
        }
    }
}

// (sigma_ij / r)^2 from 1/r^2: sigma_ij^2 from the table entry (TAB) or the two
// beads' sigma.
template <bool TAB, CoordForm FORM>
__device__ __forceinline__ float sigma2_over_r2(const float4 &et, float inv2, float si, float sj, float u2, float u2l)
{
    if (TAB) return FORM == FRACTION ? __builtin_fmaf(inv2, et.y, inv2 * et.z) : inv2 * et.y;
    const float sij = 0.5f * (si + sj), t = sij * sij * inv2;
    return FORM == FRACTION ? __builtin_fmaf(t, u2, t * u2l) : t;
}

// How far from the middle of a group of extent w (k_fix) a bead of |x| + |y| +
// |z| = size may lie to reach one of the group's beads within the crowder cutoff
// as float distances have it.  0.1 A covers the distances' own rounding; each
// difference of two coordinates is rounded by up to 2^-24 of their sizes (they
// may lie boxes away, or in a box of 1e6 A), in the pair's distance and in the
// screen's: 2^-22 of the bead's size here, of the group's in w.
constexpr float SCREEN_ROUND = 2.384185791015625e-7f; // 2^-22
__device__ __forceinline__ float screen_limit(float w, const DevFF &ff, float size)
{
    return __builtin_fmaf(size, SCREEN_ROUND, w + ff.crow_cut + 0.1f);
}

// Walks the columns of group g against the wave's rows.  op is called as
//   op.contact(j, n, charged, later)  n beads' contact pairs (beads j..) with
//       rows of other bodies; charged: bit k set where bead j + k carries a
//       charge; later: their bodies come after the rows'
//   op.masked(j, n, charged, diag)  the same, less what is no contact pair of
//       two bodies
//   op.crowder(j, diag)   bead j's crowder pairs with the rows
// and, in the diagonal tile, leaves out all pairs (op.masked, op.crowder) but
// those of a later column than row.
template <class OP>
__device__ __forceinline__ void walk_group(OP &op, const Beads &B, int g, const Row &r, bool diag, const DevSys &S,
                                           const DevFF &ff)
{
    const int b0 = B.g[4 * g], b1 = B.g[4 * g + 1], kc = B.g[4 * g + 2], chm = B.g[4 * g + 3];
    const int kinds = kc & 0xff, cnt = kc >> 8, j = g * GROUP;
    if (kinds & r.kinds & GROUP_CHAIN) {
        if (((kinds | r.kinds) & GROUP_CROWDER) == 0 && !diag && (b1 < r.b0 || b0 > r.b1) && !op.general()) {
            op.contact(j, cnt, chm, b0 > r.b1);
            return;
        }
        if (b0 != b1 || r.b0 != r.b1 || b0 != r.b0) op.masked(j, cnt, chm, diag); // else all of one body
    }
    if (((kinds | r.kinds) & GROUP_CROWDER) == 0 || !op.crowders()) return;
    if (kinds & GROUP_CROWDER) {
        // crowder columns that may reach a row: lane 16 q + k looks at column k
        // and row group q
        const int lane = threadIdx.x & 63, k = lane & 15, q = lane >> 4;
        bool near = false;
        if (k < cnt && q < r.gn && (op.tcs[j + k] >> 8) != 0) {
            const float4 c = op.gc[r.g0 + q];
            const float x = op.gx[j + k], y = op.gy[j + k], z = op.gz[j + k];
            const float lim = screen_limit(c.w, ff, fabsf(x) + fabsf(y) + fabsf(z));
            near = !(dist2(x, y, z, c, S) > lim * lim);
        }
        const unsigned long long m4 = __ballot(near);
        for (unsigned int m = (unsigned int)(m4 | m4 >> 16 | m4 >> 32 | m4 >> 48) & 0xFFFFu; m; m &= m - 1u)
            op.crowder(j + __builtin_ctz(m), diag);
    }
    if ((kinds & GROUP_CHAIN) && (r.kinds & GROUP_CROWDER)) {
        // the group's extent against the crowder rows
        const float lim = screen_limit(B.c[4 * g + 3], ff, r.size);
        const float d2 = dist2(B.c[4 * g], B.c[4 * g + 1], B.c[4 * g + 2], make_float4(r.x, r.y, r.z, 0.f), S);
        if (__any(r.crow && !(d2 > lim * lim)))
            for (int k = 0; k < cnt; ++k)
                if ((B.tc[j + k] >> 8) == 0) op.crowder(j + k, diag);
    }
}

// What the kernels below read of the conformation, made once a call:
//   fix[k * p.copy_beads + b], k = 0..2: coordinate k of replica bead b as a
//     fraction of its box (boxes of up to FIX_BOX_MAX);
//   then per replica and group of 16 beads (R.grp_off groups before the
//   replica's) the middle of the range of their coordinates and half its
//   diagonal (with what rounding may add, screen_limit), 4 floats.
__global__ __launch_bounds__(256) void k_fix(KParams p, int rep_first, int *fix)
{
    const DevRep R = p.rep[rep_first + blockIdx.y];
    const DevSys S = p.sys[R.sys];
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b - (int)(threadIdx.x & 15) >= S.n_beads) return; // whole groups
    const bool on = b < S.n_beads;
    const size_t i = (size_t)R.bead_off + min(b, S.n_beads - 1);
    const float x = p.px[i], y = p.py[i], z = p.pz[i];
    if (on && box_in_fractions(S.box)) {
        fix[i] = fix_coord(x, S.unit);
        fix[p.copy_beads + i] = fix_coord(y, S.unit);
        fix[2 * p.copy_beads + i] = fix_coord(z, S.unit);
    }
    // lanes past the last bead repeat it
    const float lx = row16<false>(x), ly = row16<false>(y), lz = row16<false>(z);
    const float hx = row16<true>(x), hy = row16<true>(y), hz = row16<true>(z);
    if ((threadIdx.x & 15) == 0) {
        const float ex = hx - lx, ey = hy - ly, ez = hz - lz;
        const float mx = fmaxf(-lx, hx), my = fmaxf(-ly, hy), mz = fmaxf(-lz, hz); // the largest sizes
        ((float4 *)(fix + fix_centres(p.copy_beads)))[(size_t)R.grp_off + b / GROUP] =
            make_float4(0.5f * (lx + hx), 0.5f * (ly + hy), 0.5f * (lz + hz),
                        0.5f * sqrtf(ex * ex + ey * ey + ez * ez) + SCREEN_ROUND * (mx + my + mz));
    }
}

static void launch_fix(const KParams &p, int rep_first, int n_rep, int max_beads, int *fix, hipStream_t s)
{
    hipLaunchKernelGGL(k_fix, dim3((max_beads + 255) / 256, n_rep), dim3(256), 0, s, p, rep_first, fix);
}

// --------------------------------------------------------------------------
// batched full energy
// --------------------------------------------------------------------------
// With T tiles of 64 beads, row tile a meets tiles a, a + 1, ..., a + T/2 (mod
// T; the last only for a < T/2 when T is even), so every unordered tile pair is
// visited once and every row tile has the same work.  A workgroup takes an even
// share of the T (T/2 + 1) column tiles and writes one FP64 partial.
// 32 x 1300 beads: 55 -> 34 us; 64 x 11000 beads: 2.64 -> 1.74 ms (39.8M contact
// pairs a replica at 25.7 VALU instructions a wave's 64 of them, one every 3.9
// cycles of a SIMD, where one takes four; 256-bead tiles staged in LDS lost a
// quarter to padding).
// A system of up to FULL_SMALL beads forms its contact pairs from float
// differences by the moves' own operations (pair_lj_dh), so that its total and
// the sums of its moves' dE are made of the same terms: a few chains that are
// apart have an energy that is what is left of terms that nearly cancel, and in
// other terms it would differ by their rounding.  The terms are no more exact,
// and it can happen at any size; the line is where that form stops being cheap.
// A launch of 8 or 32 replicas, in us, this form and the walk: 100 beads 17.9 and
// 17.4, 200 beads 18.4 and 17.5, 256 beads 19 and 16, 320 beads 19 and 16, 1300
// beads 32-70 and 26-44.
constexpr int FULL_SMALL = 256;

template <bool TAB, CoordForm FORM, bool SMALL>
struct EnergyOp {
    const Beads &B;
    const float *gx, *gy, *gz; // positions, types and groups, for reads by lane
    const int *tcs;
    const float4 *gc;
    const Row &r;
    const RowFix &f;
    const DevSys &S;
    const DevFF &ff;
    const float4 *erow; // of the row's type: 4 E_ij, sigma_ij^2 in the unit of distance squared (high and low part)
    float s;            // the row's sigma
    float qu, kdh;      // the row's charge times the Debye-Hueckel coefficient, and the exponent scale, in the unit of
                        // contact distances
    float u2, u2l;      // 1 A^2 in the unit squared (high and low part)
    float q;            // the row's charge times the Debye-Hueckel coefficient
    bool free_only;     // non-crowder pairs only
    double acc;

    __device__ __forceinline__ bool crowders() const { return !free_only; }
    __device__ __forceinline__ bool general() const { return SMALL; }
    struct Term {
        float r2, x6, e4, e;
    };
    __device__ __forceinline__ Term term(const Column &c)
    {
        Term t;
        const float4 et = erow[c.tc];
        float dx, dy, dz;
        separation<FORM>(c, r, f, S, dx, dy, dz);
        t.r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
        const float s2 = sigma2_over_r2<TAB, FORM>(et, __builtin_amdgcn_rcpf(t.r2), s, c.s, u2, u2l);
        t.x6 = s2 * s2 * s2;
        t.e4 = et.x;
        t.e = et.x * __builtin_fmaf(-t.x6, t.x6, t.x6);
        return t;
    }
    __device__ __forceinline__ void charged(Term &t, float qc)
    {
        asm volatile("" : "+v"(t.r2)); // keeps the term behind its branch
        const float rinv = __builtin_amdgcn_rsqf(t.r2);
        t.e = __builtin_fmaf(qu * qc * __builtin_amdgcn_exp2f(t.r2 * rinv * kdh), rinv, t.e);
    }
    __device__ __forceinline__ void flip(Term &t)
    {
        if (!(t.x6 <= 0.5f) && t.e4 > 0.0f) t.e = t.e4 * (__builtin_fmaf(t.x6, t.x6, -t.x6) + 0.5f);
    }
    // NC columns: independent chains, one test of the near terms
    template <int NC>
    __device__ __forceinline__ void step(const Column *c, int chm)
    {
        Term t[NC];
        bool far = true;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            t[k] = term(c[k]);
            far = far && t[k].x6 <= 0.5f; // NaN (coincident beads) is not far
        }
        if (__all(far)) {
#pragma unroll
            for (int k = 0; k < NC; ++k)
                if (chm & (1 << k)) charged(t[k], c[k].q);
        } else {
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                flip(t[k]);
                if (chm & (1 << k)) charged(t[k], c[k].q);
                t[k].e = fminf(t[k].e, 1e30f);
            }
        }
#pragma unroll
        for (int k = 0; k < NC; ++k) acc += (double)t[k].e;
    }
    __device__ __forceinline__ void contact(int j, int n, int chm, bool)
    {
        int k = 0;
        for (; k + 3 < n; k += 4) {
            Column c[4];
            load_columns<TAB, FORM, 4>(B, j + k, c);
            step<2>(c, chm >> k);
            step<2>(c + 2, chm >> (k + 2));
        }
        for (; k < n; ++k) {
            Column c;
            load_columns<TAB, FORM, 1>(B, j + k, &c);
            step<1>(&c, chm >> k);
        }
    }
    __device__ __forceinline__ void masked(int j, int n, int chm, bool diag)
    {
        for (int k = 0; k < n; ++k) {
            Column c;
            load_columns<TAB, FORM, 1>(B, j + k, &c);
            if ((c.tc >> 8) != 0) continue; // uniform
            const bool on = B.body[j + k] != r.body && !r.crow && (!diag || j + k > r.i);
            float e;
            if (SMALL) {
                const float sij = 0.5f * (s + B.s[j + k]);
                e = pair_lj_dh(dist2(B.x[j + k], B.y[j + k], B.z[j + k], make_float4(r.x, r.y, r.z, 0.f), S), erow[c.tc].x,
                               sij * sij, q * c.q, ff);
            } else {
                Term t = term(c);
                flip(t);
                if (chm & (1 << k)) charged(t, c.q);
                e = fminf(t.e, 1e30f);
            }
            acc += (double)(on ? e : 0.0f);
        }
    }
    __device__ __forceinline__ void crowder(int j, bool diag)
    {
        const float r2 = dist2(B.x[j], B.y[j], B.z[j], make_float4(r.x, r.y, r.z, 0.f), S);
        if (r2 < ff.crow_cut2 && B.body[j] != r.body && ((B.tc[j] >> 8) != 0 || r.crow) && (!diag || j > r.i))
            acc += (double)pair_crowder(r2, ff);
    }
};

// The pointers of replica R (its conformation's, with what k_fix made of it)
// and of its system S.
__device__ __forceinline__ Beads replica_beads(const KParams &p, const DevRep &R, const DevSys &S, const int *fix)
{
    const int *fx = fix + R.bead_off, *fy = fx + p.copy_beads, *fz = fy + p.copy_beads;
    return {(Uniform<float>)(p.px + R.bead_off),
            (Uniform<float>)(p.py + R.bead_off),
            (Uniform<float>)(p.pz + R.bead_off),
            (Uniform<float>)(p.q + S.bead_off),
            (Uniform<float>)(p.sig + S.bead_off),
            (Uniform<int>)(p.tc + S.bead_off),
            (Uniform<int>)(p.body + S.bead_off),
            (Uniform<int>)fx,
            (Uniform<int>)fy,
            (Uniform<int>)fz,
            (Uniform<int>)(p.grp + 4 * (size_t)S.grp_off),
            (Uniform<float>)(fix + fix_centres(p.copy_beads) + 4 * (size_t)R.grp_off)};
}

// The type table of the contact pairs in LDS: scale e_ij, sigma_ij^2 in the
// unit squared (u2) as high and low part, w_ij.
__device__ __forceinline__ void load_table(float4 *s_et, const KParams &p, int sys, const float *e, float scale, double u2,
                                           const float *w)
{
    for (int k = threadIdx.x; k < REMC_NTYPES * REMC_NTYPES; k += COLS) {
        const double s2 =
            p.sigtab ? (double)p.sstab[((size_t)2 * sys + 1) * (REMC_NTYPES * REMC_NTYPES) + k] * u2 : 0.0;
        const float hi = (float)s2;
        s_et[k + k / REMC_NTYPES] = make_float4(scale * e[k], hi, (float)(s2 - (double)hi), w ? w[k] : 0.0f);
    }
}

__global__ __launch_bounds__(COLS) void k_energy_full(KParams p, const int *fix, double *partials, int noncrowder_only)
{
    __shared__ float4 s_et[REMC_NTYPES * TSTRIDE];
    __shared__ double s_red[WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rep = blockIdx.y;
    const DevRep R = p.rep[rep];
    const DevSys S = p.sys[R.sys];
    const int N = S.n_beads, T = full_tiles(N), h = T / 2, groups = full_groups(N);
    const DevFF ff = p.ff;
    const Beads B = replica_beads(p, R, S, fix);
    const float *gx = p.px + R.bead_off, *gy = p.py + R.bead_off, *gz = p.pz + R.bead_off;
    const int *tcs = p.tc + S.bead_off, *bodies = p.body + S.bead_off;
    const double unit = S.unit, u2 = unit * unit; // of contact distances, per Angstrom
    const float u2h = (float)u2, u2l = (float)(u2 - (double)u2h);
    const float4 *gc = (const float4 *)(fix + fix_centres(p.copy_beads)) + R.grp_off;
    load_table(s_et, p, R.sys, p.etab, 1.0f, u2, nullptr);
    __syncthreads();
    // this workgroup's column tiles, of all row tiles' in order
    const long long all = (long long)T * (h + 1);
    const int u0 = (int)(all * blockIdx.x / gridDim.x), u1 = (int)(all * (blockIdx.x + 1) / gridDim.x);
    auto walk = [&](auto tab, auto form, auto small) __attribute__((always_inline)) {
        double sum = 0.0;
        for (int u = u0; u < u1;) {
            const int a = u / (h + 1), bo0 = u % (h + 1), end = min(h + 1, bo0 + (u1 - u));
            u += end - bo0;
            // the last offset of an even T belongs to one of the two tiles
            const int bo1 = min(end, T % 2 == 0 && h > 0 && a >= h ? h : h + 1);
            const Row row = load_row(a, N, gx, gy, gz, tcs, bodies);
            const int i = row.on ? row.i : N - 1;
            const RowFix rf = load_row_fix(row, fix + R.bead_off, fix + p.copy_beads + R.bead_off,
                                           fix + 2 * p.copy_beads + R.bead_off, N);
            EnergyOp<decltype(tab)::value, decltype(form)::value, decltype(small)::value> op{
                B, gx, gy, gz, tcs, gc, row, rf, S, ff, s_et + row.type * TSTRIDE, p.sig[S.bead_off + i],
                (float)((double)(p.q[S.bead_off + i] * ff.c_dh) * unit), (float)((double)ff.k_dh / unit), u2h, u2l,
                p.q[S.bead_off + i] * ff.c_dh, noncrowder_only != 0, 0.0};
            for (int k = (ROWS / GROUP) * bo0 + wave; k < (ROWS / GROUP) * bo1; k += WAVES) {
                int t = a + k / (ROWS / GROUP);
                if (t >= T) t -= T;
                const int g = t * (ROWS / GROUP) + k % (ROWS / GROUP);
                if (g < groups) walk_group(op, B, g, row, k < ROWS / GROUP, S, ff);
            }
            sum += row.on ? op.acc : 0.0;
        }
        return sum;
    };
    using T1 = std::true_type;
    using T0 = std::false_type;
    auto by_table = [&](auto form) __attribute__((always_inline)) {
        return p.sigtab ? walk(T1{}, form, T0{}) : walk(T0{}, form, T0{});
    };
    const double v = wave_sum_dpp(N <= FULL_SMALL           ? walk(T0{}, Form<FLAT>{}, T1{})
                                  : box_in_fractions(S.box) ? by_table(Form<FRACTION>{})
                                  : S.box > 0.f             ? by_table(Form<IMAGE>{})
                                                            : by_table(Form<FLAT>{}));
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < WAVES; ++w) t += s_red[w];
        partials[(size_t)rep * gridDim.x + blockIdx.x] = t;
    }
}

// one wave per replica: lane l adds workgroups l, l+64, ... in order, then a
// fixed-order wave sum (the same total on every call)
__global__ __launch_bounds__(64) void k_sum_partials(KParams p, int units, const double *partials, double *out, int write_E,
                                                     Signal sig)
{
    const int r = blockIdx.x, lane = threadIdx.x;
    double t = 0.0;
    for (int x = lane; x < units; x += 64) t += partials[(size_t)r * units + x];
    t = wave_sum_dpp(t);
    if (lane == 0) {
        if (out) host_store(out + r, t);
        if (write_E) p.E[r] = t;
    }
    signal_done(sig);
}

int full_units(int n_rep, int max_beads)
{
    const long long T = full_tiles(max_beads), all = T * (T / 2 + 1), want = (FULL_WG + n_rep - 1) / n_rep;
    const long long most = std::max(want, (all + FULL_PER_MAX - 1) / FULL_PER_MAX);
    if (most >= all) return (int)all;
    const long long per = all / most; // column tiles of a workgroup, rounded to an even share
    return (int)((all + per - 1) / per);
}

hipError_t launch_energy_full(const KParams &p, int n_rep, int max_beads, int *fix, double *partials, double *out,
                              int noncrowder_only, int write_E, hipStream_t s, const Signal &sig)
{
    if (n_rep <= 0) return hipSuccess;
    launch_fix(p, 0, n_rep, max_beads, fix, s);
    const int units = full_units(n_rep, max_beads);
    hipLaunchKernelGGL(k_energy_full, dim3(units, n_rep), dim3(COLS), 0, s, p, fix, partials, noncrowder_only);
    hipLaunchKernelGGL(k_sum_partials, dim3(n_rep), dim3(64), 0, s, p, units, partials, out, write_E, sig);
    return hipGetLastError();
}

// --------------------------------------------------------------------------
// adjoint: gradient of the full energy, every replica of a range in one launch
//
// k_adjoint_rows: one workgroup per (row tile, partner sub-range, replica); the
// lanes sum in FP64, from FP32 pair derivatives (the branches of the pair
// term), dE/dx_i of their row bead and, over the unordered pairs (those whose
// column belongs to a later body), the parameter derivatives
// dE/dlambda = sum dE/dE_ij (T_ij - e0), dE/de0 = -lambda sum dE/dE_ij and
// dE/dxi = sum DH r / xi^2.  The waves' row gradients are added through LDS in wave order and written once per
// (sub-range, bead), their parameter sums once per workgroup.
// k_adjoint_bodies: one wave per (replica, body) adds each bead's sub-range
// partials in sub-range order, forms F = -sum dE/dx_i and the torque
// sum rel_i x F_i about the body centre with fixed-order wave sums; the first
// wave of each replica adds the parameter partials.  The result does not
// depend on scheduling.  Sub-ranges are only cut when the launch holds fewer
// than ADJ_TARGET_WG (row tile, replica) workgroups.
// 32 x 1300 beads: 87 + 14 -> 70 + 6 us; 64 x 11000 beads: 8.15 + 0.06 -> 5.0 ms
// (39 VALU instructions a wave's 64 ordered pairs, one every 3.7 cycles).
// --------------------------------------------------------------------------
struct AdjFF {
    float t0[REMC_NTYPES * REMC_NTYPES]; // T_ij - e0
    float e[REMC_NTYPES * REMC_NTYPES];  // E_ij = lambda (T_ij - e0)
    float lambda, xi, c_lj, c_dh;
};

constexpr int ADJ_TARGET_WG = 2048; // workgroups a launch aims at

template <bool TAB, CoordForm FORM>
struct AdjointOp {
    const Beads &B;
    const float *gx, *gy, *gz; // positions, types and groups, for reads by lane
    const int *tcs;
    const float4 *gc;
    const Row &r;
    const RowFix &f;
    const DevSys &S;
    const DevFF &ff;
    float lambda;
    const float4 *erow; // of the row's type: 24 c_lj E_ij, sigma_ij^2 as above, T_ij - e0
    float s;            // the row's sigma
    float qu, kdh, ixu; // the row's charge times the Debye-Hueckel coefficient, the exponent scale and 1/xi in the
                        // unit of contact distances
    float u2, u2l;      // 1 A^2 in the unit squared (high and low part)
    // contact sums over the columns: derivative times (column - row) in units,
    // dE/dE_ij / (4 c_lj) times T_ij - e0 and alone, Debye-Hueckel times r in units;
    // ax.. of the other pairs in Angstrom
    double ux, uy, uz, pl, pe, px, ax, ay, az;

    __device__ __forceinline__ bool crowders() const { return true; }
    __device__ __forceinline__ bool general() const { return false; }
    struct Term {
        float dx, dy, dz, r2, inv2, x6, kf, u, t0;
    };
    // One contact pair without its charges: (dE/dr)/r in units^-2, and with PAR
    // the parameter terms.
    template <bool PAR>
    __device__ __forceinline__ Term term(const Column &c)
    {
        Term o;
        const float4 et = erow[c.tc];
        separation<FORM>(c, r, f, S, o.dx, o.dy, o.dz);
        o.r2 = fmaxf(__builtin_fmaf(o.dx, o.dx, __builtin_fmaf(o.dy, o.dy, o.dz * o.dz)), 1e-36f);
        o.inv2 = __builtin_amdgcn_rcpf(o.r2);
        const float s2 = sigma2_over_r2<TAB, FORM>(et, o.inv2, s, c.s, u2, u2l);
        o.x6 = s2 * s2 * s2;
        o.kf = et.x * o.x6 * __builtin_fmaf(2.0f, o.x6, -1.0f) * o.inv2;
        if (PAR) {
            o.t0 = et.w;
            o.u = -(o.x6 * (o.x6 - 1.0f));
        }
        return o;
    }
    template <bool PAR>
    __device__ __forceinline__ void flip(Term &o, const Column &c)
    {
        const bool f = o.x6 > 0.5f && lambda * erow[c.tc].w > 0.0f;
        o.kf = f ? -o.kf : o.kf;
        if (PAR) o.u = f ? 0.5f - o.u : o.u;
    }
    // adds the Debye-Hueckel derivative; the term itself times r
    __device__ __forceinline__ float charged(Term &o, float qc)
    {
        asm volatile("" : "+v"(o.r2)); // keeps the term behind its branch
        const float rinv = __builtin_amdgcn_rsqf(o.r2);
        const float rr = o.r2 * rinv;
        const float dh = qu * qc * __builtin_amdgcn_exp2f(rr * kdh) * rinv;
        o.kf = __builtin_fmaf(-dh * (ixu + rinv), rinv, o.kf);
        return dh * rr;
    }
    // A pair's products are formed and added in FP64 (an FMA each: seven
    // instructions for the force, against nine for FP32 products added in FP64).
    __device__ __forceinline__ void add_force(const Term &t)
    {
        const double k = (double)t.kf;
        ux = __builtin_fma(k, (double)t.dx, ux);
        uy = __builtin_fma(k, (double)t.dy, uy);
        uz = __builtin_fma(k, (double)t.dz, uz);
    }
    __device__ __forceinline__ void add_params(const Term &t)
    {
        const double u = (double)t.u;
        pl = __builtin_fma(u, (double)t.t0, pl);
        pe += u;
    }
    template <bool PAR>
    __device__ __forceinline__ void add_charge(float dhr)
    {
        if (PAR) px += (double)dhr;
    }
    // two columns: independent chains, one test of the near terms
    template <bool PAR>
    __device__ __forceinline__ void two(const Column *c, int ch)
    {
        Term a = term<PAR>(c[0]), b = term<PAR>(c[1]);
        if (__any(a.x6 > 0.5f || b.x6 > 0.5f)) {
            flip<PAR>(a, c[0]);
            flip<PAR>(b, c[1]);
        }
        if (ch & 1) add_charge<PAR>(charged(a, c[0].q));
        if (ch & 2) add_charge<PAR>(charged(b, c[1].q));
        add_force(a);
        add_force(b);
        if (PAR) {
            add_params(a);
            add_params(b);
        }
    }
    template <bool PAR>
    __device__ __forceinline__ void contacts(int j, int n, int chm)
    {
        int k = 0;
        for (; k + 3 < n; k += 4) {
            Column c[4];
            load_columns<TAB, FORM, 4>(B, j + k, c);
            two<PAR>(c, chm >> k);
            two<PAR>(c + 2, chm >> (k + 2));
        }
        for (; k < n; ++k) {
            Column c;
            load_columns<TAB, FORM, 1>(B, j + k, &c);
            Term a = term<PAR>(c);
            if (__any(a.x6 > 0.5f)) flip<PAR>(a, c);
            if ((chm >> k) & 1) add_charge<PAR>(charged(a, c.q));
            add_force(a);
            if (PAR) add_params(a);
        }
    }
    __device__ __forceinline__ void contact(int j, int n, int chm, bool later)
    {
        if (later) // each unordered pair once for the parameter sums
            contacts<true>(j, n, chm);
        else
            contacts<false>(j, n, chm);
    }
    __device__ __forceinline__ void masked(int j, int n, int chm, bool)
    {
        for (int k = 0; k < n; ++k) {
            Column c;
            load_columns<TAB, FORM, 1>(B, j + k, &c);
            if ((c.tc >> 8) != 0) continue; // uniform
            const int body = B.body[j + k];
            Term a = term<true>(c);
            flip<true>(a, c);
            const float dhr = (chm >> k) & 1 ? charged(a, c.q) : 0.0f;
            if (body != r.body && !r.crow) {
                add_force(a);
                if (body > r.body) { // each unordered pair once for the parameter sums
                    add_params(a);
                    add_charge<true>(dhr);
                }
            }
        }
    }
    __device__ __forceinline__ void crowder(int j, bool)
    {
        const float dx = min_image(B.x[j] - r.x, S.box, S.inv_box), dy = min_image(B.y[j] - r.y, S.box, S.inv_box),
                    dz = min_image(B.z[j] - r.z, S.box, S.inv_box);
        const float r2 = fmaxf(__builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)), 1e-36f);
        if (r2 < ff.crow_cut2 && B.body[j] != r.body && ((B.tc[j] >> 8) != 0 || r.crow)) {
            const float rinv = __builtin_amdgcn_rsqf(r2);
            const float t = ff.crow_s2 * (rinv * rinv);
            const float t6 = t * t * t;
            const float kf = -6.0f * ff.c_crow * t6 * rinv * rinv;
            ax += (double)(kf * dx);
            ay += (double)(kf * dy);
            az += (double)(kf * dz);
        }
    }
};

// (6 waves a SIMD: 80 registers)
__global__ __launch_bounds__(COLS, 6) void k_adjoint_rows(KParams p, AdjFF af, int rep_first, int tiles, int split,
                                                          int sub_len, int bead_base, size_t bead_stride, const int *fix,
                                                          double *part_grad, double *param_part)
{
    __shared__ float4 s_et[REMC_NTYPES * TSTRIDE];
    __shared__ double s_g[WAVES - 1][3][ROWS];
    __shared__ double s_pp[WAVES][3];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = blockIdx.x / split, sub = blockIdx.x % split;
    const int rr = blockIdx.y;
    const DevRep R = p.rep[rep_first + rr];
    const DevSys S = p.sys[R.sys];
    const DevFF ff = p.ff;
    const int N = S.n_beads;
    const int j0 = sub * sub_len;
    if (tile * ROWS >= N || j0 >= N) return; // the whole workgroup, before any barrier
    const int j1 = min(N, j0 + sub_len);
    const Beads B = replica_beads(p, R, S, fix);
    const float *gx = p.px + R.bead_off, *gy = p.py + R.bead_off, *gz = p.pz + R.bead_off;
    const double unit = S.unit, u2 = unit * unit; // of contact distances, per Angstrom
    const float u2h = (float)u2, u2l = (float)(u2 - (double)u2h);
    const float4 *gc = (const float4 *)(fix + fix_centres(p.copy_beads)) + R.grp_off;
    load_table(s_et, p, R.sys, af.e, 24.0f * af.c_lj, u2, af.t0);
    const Row row = load_row(tile, N, gx, gy, gz, p.tc + S.bead_off, p.body + S.bead_off);
    const int i = row.on ? row.i : N - 1;
    const RowFix rf = load_row_fix(row, fix + R.bead_off, fix + p.copy_beads + R.bead_off,
                                   fix + 2 * p.copy_beads + R.bead_off, N);
    __syncthreads();
    double g[3], v[3];
    const float lambda = af.lambda, xi = af.xi, c_lj = af.c_lj, c_dh = af.c_dh;
    auto walk = [&](auto tab, auto form) __attribute__((always_inline)) {
        AdjointOp<decltype(tab)::value, decltype(form)::value> op{
            B, gx, gy, gz, p.tc + S.bead_off, gc, row, rf, S, ff, lambda, s_et + row.type * TSTRIDE, p.sig[S.bead_off + i],
            (float)((double)(p.q[S.bead_off + i] * c_dh) * unit), (float)((double)ff.k_dh / unit),
            (float)(1.0 / ((double)xi * unit)), u2h, u2l, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int k = j0 / GROUP + wave; k < (j1 + GROUP - 1) / GROUP; k += WAVES) walk_group(op, B, k, row, false, S, ff);
        // column minus row: dE/dx_i is minus the sum; (dE/dr)/r times a
        // difference, both in units, is dE/dr per unit
        g[0] = -(op.ux * unit + op.ax);
        g[1] = -(op.uy * unit + op.ay);
        g[2] = -(op.uz * unit + op.az);
        const double scale = 4.0 * (double)c_lj;
        v[0] = wave_sum_dpp(row.on ? scale * op.pl : 0.0);
        v[1] = wave_sum_dpp(row.on ? -scale * (double)lambda * op.pe : 0.0);
        v[2] = wave_sum_dpp(row.on ? op.px / (unit * (double)xi * (double)xi) : 0.0);
    };
    auto by_table = [&](auto form) __attribute__((always_inline)) {
        p.sigtab ? walk(std::true_type{}, form) : walk(std::false_type{}, form);
    };
    if (box_in_fractions(S.box))
        by_table(Form<FRACTION>{});
    else if (S.box > 0.f)
        by_table(Form<IMAGE>{});
    else
        by_table(Form<FLAT>{});
    if (wave > 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) s_g[wave - 1][k][lane] = g[k];
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) s_pp[wave][k] = v[k];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < WAVES - 1; ++w)
            for (int k = 0; k < 3; ++k) g[k] += s_g[w][k][lane];
        if (row.on) {
            double *pg = part_grad + 3 * ((size_t)sub * bead_stride + (size_t)(R.bead_off - bead_base) + i);
            pg[0] = g[0];
            pg[1] = g[1];
            pg[2] = g[2];
        }
        if (lane < 3) {
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) t += s_pp[w][lane];
            param_part[3 * (((size_t)rr * tiles + tile) * split + sub) + lane] = t;
        }
    }
}

// One wave per (replica, body of several beads): the lanes stride over the
// body's beads, then wave sums (fixed order, so every call gives the same
// bits); one lane per (replica, one-bead body) after them (p.border: the
// bodies in that order), where a wave each kept one lane of 64 busy.  The first
// wave of each replica also adds its parameter partials.
__global__ __launch_bounds__(256) void k_adjoint_bodies(KParams p, int rep_first, int tiles, int split, int sub_len,
                                                        int bead_base, size_t bead_stride, int body_base,
                                                        const double *part_grad, const double *param_part,
                                                        double *force_torque, double *dparams)
{
    const int rr = blockIdx.y;
    const DevRep R = p.rep[rep_first + rr];
    const DevSys S = p.sys[R.sys];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int N = S.n_beads;
    const int nsub = (N + sub_len - 1) / sub_len, ntile = (N + ROWS - 1) / ROWS;
    if (blockIdx.x == 0 && wave == 0) {
        double t0 = 0.0, t1 = 0.0, t2 = 0.0;
        for (int a = lane; a < ntile * nsub; a += 64) {
            const int tile = a / nsub, sub = a - tile * nsub;
            const double *pp = param_part + 3 * (((size_t)rr * tiles + tile) * split + sub);
            t0 += pp[0];
            t1 += pp[1];
            t2 += pp[2];
        }
        t0 = wave_sum_dpp(t0);
        t1 = wave_sum_dpp(t1);
        t2 = wave_sum_dpp(t2);
        if (lane == 0) {
            dparams[3 * rr + 0] = t0;
            dparams[3 * rr + 1] = t1;
            dparams[3 * rr + 2] = t2;
        }
    }
    const int w = blockIdx.x * (blockDim.x >> 6) + wave;
    const bool several = w < S.n_multi;
    const int o = several ? w : S.n_multi + (w - S.n_multi) * 64 + lane;
    if (o >= S.n_bodies) return;
    const int m = p.border[S.body_off + o];
    const int b0 = p.bstart[S.body_off + m], b1 = p.bend[S.body_off + m];
    const float *rx = p.rx + R.bead_off, *ry = p.ry + R.bead_off, *rz = p.rz + R.bead_off;
    const double *pg = part_grad + 3 * (size_t)(R.bead_off - bead_base);
    double F[3] = {0.0, 0.0, 0.0}, T[3] = {0.0, 0.0, 0.0};
    for (int i = several ? b0 + lane : b0; i < b1; i += 64) {
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        for (int s = 0; s < nsub; ++s) {
            const double *q = pg + 3 * ((size_t)s * bead_stride + i);
            g0 += q[0];
            g1 += q[1];
            g2 += q[2];
        }
        const double f0 = -g0, f1 = -g1, f2 = -g2;
        F[0] += f0; F[1] += f1; F[2] += f2;
        const double ax = rx[i], ay = ry[i], az = rz[i];
        T[0] += ay * f2 - az * f1;
        T[1] += az * f0 - ax * f2;
        T[2] += ax * f1 - ay * f0;
    }
    if (several)
        for (int k = 0; k < 3; ++k) {
            F[k] = wave_sum_dpp(F[k]);
            T[k] = wave_sum_dpp(T[k]);
        }
    if (lane == 0 || !several) {
        double *out = force_torque + 6 * ((size_t)(R.body_off - body_base) + m);
        for (int k = 0; k < 3; ++k) {
            out[k] = F[k];
            out[3 + k] = T[k];
        }
    }
}

AdjPlan adjoint_plan(int n_rep, int max_beads, size_t bead_stride, int target_wg)
{
    AdjPlan a{};
    a.tiles = (max_beads + ROWS - 1) / ROWS;
    const long long target = target_wg > 0 ? target_wg : ADJ_TARGET_WG;
    const long long units = (long long)n_rep * a.tiles;
    const long long want = units >= target ? 1 : (target + units - 1) / units;
    const long long per = (max_beads + want - 1) / want;
    a.sub_len = (int)std::max<long long>(ROWS, (per + ROWS - 1) / ROWS * ROWS);
    a.split = (max_beads + a.sub_len - 1) / a.sub_len;
    a.part_doubles = 3 * (size_t)a.split * bead_stride;
    a.param_doubles = 3 * (size_t)n_rep * a.tiles * a.split;
    return a;
}

hipError_t launch_adjoint(const KParams &p, const void *adj_ff, const AdjPlan &a, int rep_first, int n_rep,
                          int max_beads, int body_waves, int bead_base, size_t bead_stride, int body_base, int *fix,
                          double *scratch, double *force_torque, double *dparams, hipStream_t s)
{
    if (n_rep <= 0) return hipSuccess;
    launch_fix(p, rep_first, n_rep, max_beads, fix, s);
    double *part_grad = scratch, *param_part = scratch + a.part_doubles;
    const AdjFF af = *(const AdjFF *)adj_ff;
    hipLaunchKernelGGL(k_adjoint_rows, dim3(a.tiles * a.split, n_rep), dim3(COLS), 0, s, p, af, rep_first,
                       a.tiles, a.split, a.sub_len, bead_base, bead_stride, fix, part_grad, param_part);
    hipLaunchKernelGGL(k_adjoint_bodies, dim3((body_waves + 3) / 4, n_rep), dim3(256), 0, s, p, rep_first, a.tiles,
                       a.split, a.sub_len, bead_base, bead_stride, body_base, part_grad, param_part, force_torque,
                       dparams);
    return hipGetLastError();
}

size_t adjoint_ff_size() { return sizeof(AdjFF); }

void adjoint_ff_fill(void *dst, const float *table, double lambda, double e0, double xi, double c_lj, double c_dh)
{
    AdjFF *a = (AdjFF *)dst;
    a->lambda = (float)lambda;
    for (int k = 0; k < REMC_NTYPES * REMC_NTYPES; ++k) {
        a->t0[k] = table[k] - (float)e0;
        a->e[k] = a->lambda * a->t0[k];
    }
    a->xi = (float)xi;
    a->c_lj = (float)c_lj;
    a->c_dh = (float)c_dh;
}

} // namespace remc
