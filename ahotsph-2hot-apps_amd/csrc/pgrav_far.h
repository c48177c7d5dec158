// Which list entries a sink group takes through its local expansion (k_far,
// pgrav_far.hip).  The Ewald kernel decides again for itself, from the same FP64
// operations, spelled out as fused multiply-adds so that both kernels round alike.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pgrav {

// A cell is far when the group's sinks reach less than FAR_RHO of its distance from the
// group centre and (eps / distance)^2 is below FAR_ETA.  At the outermost sink and for the
// nearest far cell the degrees left out are then 7.7e-6 of a point's pull; a cell's moment
// of order k brings them with a factor (l + k)! / (k! l!) (extent / distance)^k, so that a
// cell of two bodies 0.2, 0.4, 0.5 of its distance from their mean is at worst 2.6e-5,
// 7.9e-5, 1.2e-4 of m / d^2 off at order 2 and 3.5e-5, 2.3e-4, 5.0e-4 at order 4 (which
// itself leaves out the cell's order 5, (extent / distance)^5).  Most far cells are much
// farther and rounder: over all sinks the error against the FP64 evaluation of the same
// lists is below that of the pairs alone: median |da|/|a| 6.9e-8 (pairs 1.0e-7), 99th
// percentile 4.7e-7 (5.5e-7), largest 4.7e-6 of the rms pull (4.7e-6) at 1 M clustered
// bodies; on the 64^3 lattice of explicit images 1.6e-5 (5.3e-5), 9e-5 (3.1e-4), 4.9e-5
// (2.1e-4); over 70 plans of 30,000 to 700,000 bodies (orders, softenings, angles, periodic
// schemes) the 2-norm of the error is 0.8 of the pairs' in the mean and 1.002 at most, the
// largest error 1.16 at most.  0.25 gains 3 % and triples the 99th percentile; 0.15 costs
// 1.5 to 3 % (16.8 M 27.1 ms, images 64^3 813 us instead of 26.6 and 783), 0.13 3 to 8 %.
constexpr double FAR_RHO = 0.17;
constexpr double FAR_ETA = 1e-4;
// Lists a wave would not fill once stay in pairs; a group with fewer cells has no expansion
// (its sums over the lanes and its evaluation cost as much as ~30 order-4 cells).
constexpr int FAR_MIN_LIST = 32, FAR_MIN_CELLS = 64;
// The coefficients' unit of length is the sinks' radius, in FP32: below this a cell's first
// degrees, mass / d (radius / d)^l, and the radius itself leave its range.
constexpr double FAR_MIN_RADIUS = 1e-20;

// a list entry's position: bodies and cells, at the image (i, j, k) of nln/mac.c:91-111
// where lists carry one
template <int PER>
__device__ __forceinline__ double4 entry_position(const double4 *__restrict__ pos, uint32_t e,
                                                  const uint8_t *__restrict__ img, int64_t at,
                                                  int img_f, double box) {
    double4 s = pos[e];
    if (PER == 2) {
        const int im = img[at], f = img_f, hf = f >> 1;
        s.x = fma((double)(im / (f * f) - hf), box, s.x);
        s.y = fma((double)((im / f) % f - hf), box, s.y);
        s.z = fma((double)(im % f - hf), box, s.z);
    }
    return s;
}

// its offset from the group centre (PER 1: the nearest image's; by a product with
// 1 / box, not a division: a source exactly half a box away is a tie either way)
template <int PER>
__device__ __forceinline__ double3 entry_offset(double4 s, double4 gc, double box, double ibox) {
    double3 d = make_double3(s.x - gc.x, s.y - gc.y, s.z - gc.z);
    if (PER == 1) {
        d.x = fma(-box, rint(d.x * ibox), d.x);
        d.y = fma(-box, rint(d.y * ibox), d.y);
        d.z = fma(-box, rint(d.z * ibox), d.z);
    }
    return d;
}

// PER 1: the source enters the group's expansion of the Ewald correction: every sink
// sees the centre's image of it, and its other images are far against the group radius
__device__ __forceinline__ bool ewald_expands(double3 d, double4 gc, double box, double ewratio) {
    const double am = fmax(fabs(d.x), fmax(fabs(d.y), fabs(d.z)));
    return am < 0.5 * box - gc.w && gc.w <= ewratio * (box - am);
}

// far2: the square of the group's far distance (infinite: no expansion)
template <int PER>
__device__ __forceinline__ bool entry_far(double3 d, double far2, double4 gc, double box,
                                          double ewratio) {
    return fma(d.x, d.x, fma(d.y, d.y, d.z * d.z)) > far2 &&
           (PER != 1 || ewald_expands(d, gc, box, ewratio));
}

}  // namespace pgrav
