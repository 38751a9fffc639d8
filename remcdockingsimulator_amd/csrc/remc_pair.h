// remc_pair.h -- pair terms and wave reductions shared by the kernels.
//
// Pair term (Replica.cpp:584-600,694-733; CudaFunctions.cu:430-452,536-649):
// minimum image, r = |d|; crowder pairs c*(6/r)^6 for r < 15; else
// E_ij*(...) contact term with the repulsive flip plus Debye-Hueckel.
#pragma once

#include "remc_internal.h"

namespace remc {

__device__ __forceinline__ float min_image(float d, float box, float inv_box)
{
    return __builtin_fmaf(-box, __builtin_rintf(d * inv_box), d);
}

// Energy of one non-crowder pair from squared distance.  eij4 = 4 E_ij (the
// table holds the factor 4, so LJ = E (4 x6 (x6 - 1)) costs one FMA: scaling by
// 4 is exact, the result is the same bits as forming 4 x6 (x6 - 1) and E).
// SKIP_UNCHARGED: the Debye-Hueckel term is formed under a branch on qq != 0.
// Four residue types of twenty carry a charge, so where the charge product
// is the same for a whole wave (one partner bead per wave in the full energy,
// one moved bead per wave in the MC pair loops) most waves skip the exp2 and
// its multiplies.  The skipped term is +-0, so the sum is the same number;
// coincident beads still give NaN from the LJ part (r2 = 0: rinv = inf,
// x6 = inf, inf*inf - inf) and hence the 1e30 cap.  The plain per-replica
// kernel forms every term.
template <bool SKIP_UNCHARGED = true>
__device__ __forceinline__ float pair_lj_dh(float r2, float eij4, float sij2, float qq, const DevFF &ff)
{
    float rinv = __builtin_amdgcn_rsqf(r2);
    float s2 = sij2 * (rinv * rinv);
    float x6 = s2 * s2 * s2;
    float base = __builtin_fmaf(x6, x6, -x6);           // x6 (x6 - 1)
    bool flip = (eij4 > 0.0f) & (x6 > 0.5f);            // r < 2^(1/6) sigma
    float e = eij4 * (flip ? base + 0.5f : -base);      // E (LJ + 2) when flipped, else -E LJ
    if (!SKIP_UNCHARGED || qq != 0.0f) {
        float r = r2 * rinv;
        // keeps the exp2 inside the branch (otherwise it is hoisted above it
        // and the branch becomes a select)
        if (SKIP_UNCHARGED) asm volatile("" : "+v"(r));
        e = e + qq * __builtin_amdgcn_exp2f(r * ff.k_dh) * rinv;
    }
    // coincident beads (r2 = 0: rinv = inf, r = 0 * inf) give NaN; the cap
    // (IEEE minNum returns the number) turns it, like any overflow, into 1e30
    // so compensated sums stay finite
    return fminf(e, 1e30f);
}

// Crowder term C (sigma_c / r)^6 inside the cutoff as crow_k (1/r^2)^3.  r2 = 0
// (coincident beads) gives inf, capped like the pair term; no clamp is needed
// since no zero multiplies the infinity.
__device__ __forceinline__ float pair_crowder(float r2, const DevFF &ff)
{
    const float rc = __builtin_amdgcn_rcpf(r2);
    const float rc3 = rc * rc * rc;
    return r2 < ff.crow_cut2 ? fminf(ff.crow_k * rc3, 1e30f) : 0.0f;
}

__device__ __forceinline__ float dist2(float xj, float yj, float zj, float4 a, const DevSys &S)
{
    const float dx = min_image(xj - a.x, S.box, S.inv_box);
    const float dy = min_image(yj - a.y, S.box, S.inv_box);
    const float dz = min_image(zj - a.z, S.box, S.inv_box);
    return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
}

// A coordinate as a 32-bit fraction of the box (unit = 2^32/L units per
// Angstrom), modulo 1: the difference of two, taken in 32 bits, wraps to the
// nearest image.  x unit + 1.5 2^52 has a unit of 1 in its last place, so the
// low word of the sum is x unit rounded to a whole number, modulo 2^32 (for any
// |x| < 2^19 boxes).
__device__ __forceinline__ int fix_coord(float x, double unit)
{
    return __double2loint(__builtin_fma((double)x, unit, 6755399441055744.0));
}

// 64-bit DPP move of a double (both halves with the same control word).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_f64(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int l2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROW_MASK, 0xf, true);
    const int h2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROW_MASK, 0xf, true);
    return __hiloint2double(h2, l2);
}

// Sum over the 64 lanes of a wave in a fixed order, with DPP row shifts and
// row broadcasts (no LDS traffic); the result is uniform.
__device__ __forceinline__ double wave_sum_dpp(double v)
{
    v += dpp_f64<0x111, 0xf>(v); // row_shr:1
    v += dpp_f64<0x112, 0xf>(v); // row_shr:2
    v += dpp_f64<0x114, 0xf>(v); // row_shr:4
    v += dpp_f64<0x118, 0xf>(v); // row_shr:8: lane 15 of each row holds the row sum
    v += dpp_f64<0x142, 0xa>(v); // row_bcast:15: rows 1 and 3 add the previous row's sum
    v += dpp_f64<0x143, 0xc>(v); // row_bcast:31: rows 2 and 3 add lane 31
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
    return __hiloint2double(hi, lo);
}

} // namespace remc
