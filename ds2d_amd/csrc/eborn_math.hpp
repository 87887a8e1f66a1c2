// Arithmetic of the plain elastic Born pair, shared by its per-cell kernels
// and its tile kernels (device code).  Every contraction is spelled out, so
// the two round alike.
#pragma once
#include "common.hpp"

// nothing beyond the fma_ below is contracted in the files that include this
#pragma clang fp contract(off)

namespace ds2d {
namespace ebm {

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// c1 (a1 - b1) + c2 (a2 - b2) + c3 (a3 - b3) + c4 (a4 - b4), in the order of taps (wave.hpp)
__device__ __forceinline__ float diff8(float a1, float b1, float a2, float b2, float a3, float b3, float a4, float b4) {
    float s = DS2D_C1 * (a1 - b1);
    s = fma_(DS2D_C2, a2 - b2, s);
    s = fma_(DS2D_C3, a3 - b3, s);
    return fma_(DS2D_C4, a4 - b4, s);
}
// a x + b y
__device__ __forceinline__ float two(float a, float x, float b, float y) { return fma_(a, x, b * y); }

struct Moduli {
    float l, mu, l2m;
    __device__ __forceinline__ Moduli(float lam, float mu_) : l(lam), mu(mu_), l2m(lam + 2 * mu_) {}
};
// Born source of the strains on top of a stress (add_born_source, born.cu:351-405)
__device__ __forceinline__ void born_source(const Moduli& m, float dmp, float dms, float exx, float ezz, float exz,
                                            float& xx, float& zz, float& xz) {
    const float p = 2 * m.l2m * -dmp, q = 2 * fma_(m.l2m, -dmp, 2 * m.mu * dms);
    xx += two(p, exx, q, ezz);
    zz += two(q, exx, p, ezz);
    xz = fma_(2 * m.mu * -dms, exz, xz);
}
// stress increments of the velocity differences (dvx/dx, dvz/dz, dvx/dz, dvz/dx)
__device__ __forceinline__ float inc_xx(const Moduli& m, float ax, float az, float dvx, float dvz) {
    return two(ax * m.l2m, dvx, az * m.l, dvz);
}
__device__ __forceinline__ float inc_zz(const Moduli& m, float ax, float az, float dvx, float dvz) {
    return two(ax * m.l, dvx, az * m.l2m, dvz);
}
__device__ __forceinline__ float inc_xz(const Moduli& m, float ax, float az, float dvzx, float dvxz) {
    return m.mu * two(ax, dvzx, az, dvxz);
}
// imaging products of a step
__device__ __forceinline__ void image(const Moduli& m, float exx, float ezz, float exz, float xx, float zz, float xz,
                                      float& gpp, float& gps) {
    gpp = fma_(-2 * m.l2m * (exx + ezz), xx + zz, gpp);
    gps += fma_(-2 * m.mu * exz, xz, 4 * m.mu * two(ezz, xx, exx, zz));
}

}  // namespace ebm
}  // namespace ds2d
