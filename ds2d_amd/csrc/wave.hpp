// Eight-point staggered differences for one wave of 64 consecutive z cells
// (device code): the z neighbours of a lane's cell are the lanes beside it,
// reached by wave shifts, so no LDS and no barrier is needed.  The four lanes
// at either end of the wave get zeros shifted in and are halo.
#pragma once
#include "common.hpp"

namespace ds2d {

template <typename T>
struct C8;
template <>
struct C8<float> {
    static constexpr float c1 = DS2D_C1, c2 = DS2D_C2, c3 = DS2D_C3, c4 = DS2D_C4;
};
template <>
struct C8<double> {
    static constexpr double c1 = DS2D_C1, c2 = DS2D_C2, c3 = DS2D_C3, c4 = DS2D_C4;
};

// The value of the next (previous) lane: the cell below (above).
__device__ __forceinline__ float next_z(float f) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float prev_z(float f) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double next_z(double f) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(f), 0x130, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(f), 0x130, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double prev_z(double f) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(f), 0x138, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(f), 0x138, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// c1 (a1 - b1) + c2 (a2 - b2) + c3 (a3 - b3) + c4 (a4 - b4)
template <typename T>
__device__ __forceinline__ T taps(T a1, T b1, T a2, T b2, T a3, T b3, T a4, T b4) {
    return fma(C8<T>::c4, a4 - b4, fma(C8<T>::c3, a3 - b3, fma(C8<T>::c2, a2 - b2, C8<T>::c1 * (a1 - b1))));
}
// Forward and backward half-point differences along z.
template <typename T>
__device__ __forceinline__ T dplus_z(T f) {
    const T p1 = next_z(f), p2 = next_z(p1), p3 = next_z(p2), p4 = next_z(p3);
    const T m1 = prev_z(f), m2 = prev_z(m1), m3 = prev_z(m2);
    return taps(p1, f, p2, m1, p3, m2, p4, m3);
}
template <typename T>
__device__ __forceinline__ T dminus_z(T f) {
    const T p1 = next_z(f), p2 = next_z(p1), p3 = next_z(p2);
    const T m1 = prev_z(f), m2 = prev_z(m1), m3 = prev_z(m2), m4 = prev_z(m3);
    return taps(f, m1, p1, m2, p2, m3, p3, m4);
}
// Weight of the cell at offset d in a forward half-point difference.
template <typename T>
__device__ __forceinline__ T src_tap(int d) {
    return d == 1 ? C8<T>::c1 : d == 2 ? C8<T>::c2 : d == 3 ? C8<T>::c3 : d == 4 ? C8<T>::c4 :
           d == 0 ? -C8<T>::c1 : d == -1 ? -C8<T>::c2 : d == -2 ? -C8<T>::c3 : d == -3 ? -C8<T>::c4 : T(0);
}

// Rows a wave owns: the velocity and the stress (or pressure) of a step each
// use four of the eight halo rows on either side.
constexpr int WAVE_HALO = 8, WAVE_ROWS = 64 - 2 * WAVE_HALO;

}  // namespace ds2d
