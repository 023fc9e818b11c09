// physics_dev.hpp -- device helpers shared by the physics and fused kernels.
#pragma once

#include "internal.hpp"

namespace laps {

// square root in the arithmetic R of cfl_rate: correctly rounded in FP64; the
// hardware square root (about 1 ulp) in FP32; negative arguments give NaN
template <typename R>
__device__ __forceinline__ R cfl_sqrt(R x) {
    if constexpr (sizeof(R) == 4) return __builtin_amdgcn_sqrtf(x);
    else return sqrt(x);
}

// reciprocal in the arithmetic R of cfl_rate: correctly rounded in FP64; the hardware reciprocal
// (1 ulp) in FP32
template <typename R>
__device__ __forceinline__ R cfl_rcp(R x) {
    if constexpr (sizeof(R) == 4) return __builtin_amdgcn_rcpf(x);
    else return R(1) / x;
}

// Factors of cfl_rate that are the same for every point: 1/dx, 1/(dy rr), 1/(dz rr), and
// d_i / (least of dx, dy, dz) (0 without Hall); rr = R/R0.
template <typename R>
struct CflFactors {
    R ix, iy, iz, hall;
    __device__ __forceinline__ CflFactors(const PhysParams& pp, double rr) {
        double dmin = pp.dx < pp.dy ? pp.dx : pp.dy;
        if (pp.dz < dmin) dmin = pp.dz;
        ix = R(1.0 / pp.dx);
        iy = R(1.0 / (pp.dy * rr));
        iz = R(1.0 / (pp.dz * rr));
        hall = pp.hall ? R(pp.di / dmin) : R(0);
    }
};

// 1/dt of one point (vardt, mhd.f90:355-409): the caller takes the largest and inverts it once. R =
// double follows the reference's FP64 arithmetic; the mixed-precision step evaluates it in FP32
// (R = float), where the fields themselves are FP32. The reference takes per
// axis the largest of |u +- c_f|, |u +- c_s|, |u +- c_a| and |u|; with
// c_f >= c_a, c_s >= 0 (the fast speed bounds the others) that is |u| + c_f,
// which is what is computed here (equal up to the rounding of c_f against c_a
// in degenerate states, a few ulp of dt). Six square roots and one reciprocal a point; with a
// quotient for every speed and step and the square root of rho (seven and twelve) the minimum cost
// the x pass 134 us at 256^3 in FP64 (2/3 rule; 525 without it), so 77.
template <typename R>
__device__ __forceinline__ R cfl_rate(R rho, R Bx, R By, R Bz, R p, R ux, R uy, R uz, const PhysParams& pp,
                                      const CflFactors<R>& f) {
    const R zero = R(0), half = R(0.5);
    // a negative density makes the speeds NaN, as its square root would; the point then only counts
    // through the Hall speed
    const R ir = cfl_rcp(rho), ia = rho < zero ? R(__builtin_nanf("")) : ir;
    const R cs2 = R(pp.gamma) * p * ir;
    const R ax = Bx * Bx * ia, ay = By * By * ia, az = Bz * Bz * ia;
    const R cms2 = cs2 + (ax + ay + az);
    const R q = cms2 * cms2, s4 = R(4) * cs2;
    const R cnx = cfl_sqrt(fmax(q - s4 * ax, zero));
    const R cny = cfl_sqrt(fmax(q - s4 * ay, zero));
    const R cnz = cfl_sqrt(fmax(q - s4 * az, zero));
    const R cfx = cfl_sqrt(half * (cms2 + cnx)), cfy = cfl_sqrt(half * (cms2 + cny));
    const R cfz = cfl_sqrt(half * (cms2 + cnz));
    R cmx = fabs(ux) + cfx, cmy = fabs(uy) + cfy, cmz = fabs(uz) + cfz;
    if (pp.hall) {
        R bmax = Bx;  // signed max of the components (mhd.f90:396-398)
        if (By > bmax) bmax = By;
        if (Bz > bmax) bmax = Bz;
        const R ch = f.hall * ir * bmax;
        cmx = fmax(cmx, ch);
        cmy = fmax(cmy, ch);
        cmz = fmax(cmz, ch);
    }
    return fmax(fmax(cmx * f.ix, cmy * f.iy), cmz * f.iz);
}

// dt of the largest rate of some points, a non-negative double or +Inf (no finite rate)
__device__ __forceinline__ double cfl_dt(double rate) { return 1.0 / fmax(rate, 0.0); }

// k_square: grid_initialize form until the first evolve_radius, then
// update_ksquare (mhdinit.f90:114-122; AEBmod.f90:87-125); wave numbers w*
// r0r = R0/R, formed once per work-item (the reference's (k*R0)/R per mode, within an ulp)
__device__ __forceinline__ double ksquare(double kx, double ky, double kz, const PhysParams& pp, const Ctl* ctl,
                                          double r0r) {
    if (!ctl->ksq_updated) return kx * kx + ky * ky + kz * kz;
    if (pp.corot_ksq) {
        const double c = pp.cos_c, s = pp.sin_c;
        const double a = s * r0r, b = c * r0r, z = kz * r0r;
        return kx * kx * (c * c + a * a) + ky * ky * (s * s + b * b) + kx * ky * 2 * c * s * (1 - r0r * r0r) + z * z;
    }
    const double a = ky * r0r, b = kz * r0r;
    return kx * kx + a * a + b * b;
}

}  // namespace laps
