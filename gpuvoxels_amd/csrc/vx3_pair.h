// vx3_pair.h -- the geometry of a contact pair, for the kernels and for host code.
#ifndef VX3_PAIR_H
#define VX3_PAIR_H

namespace vx3 {

// The distance at which two voxels touch: 1.25 times the mean of their sizes, in the steps of
// CVX_Collision (VX_Collision.cpp:41-56); tfi, tfj: thermal factors.
template <typename real> __attribute__((always_inline)) constexpr float pairDistance(float tfi, float tfj, real nom) {
    const real b1 = nom * (real)tfi, b2 = nom * (real)tfj;
    return (float)(((b1 + b1 + b1) / (real)3.0f + (b2 + b2 + b2) / (real)3.0f) * (real)0.625f);
}

// True only for pairs whose contact force is zero (pairContact's rel <= 0), without its square
// root and divisions: most watched pairs most of the time.  The margin covers the rounding of
// the contact distance and of the length (a few parts in 2^24); a distance whose square may have
// lost bits to underflow decides nothing, nor does a NaN.
template <typename real>
__attribute__((always_inline)) constexpr bool pairApart(real xi, real yi, real zi, real xj, real yj, real zj, float tfi, float tfj, real nom) {
    const float ox = (float)(xj - xi), oy = (float)(yj - yi), oz = (float)(zj - zi);
    const float reach = (float)nom * (tfi + tfj) * 0.625f, r2 = reach * reach;
    return ox * ox + oy * oy + oz * oz > r2 * (1.0f + 0x1p-18f) && r2 > 1e-30f;
}

}  // namespace vx3
#endif
