// Lanes of the tile kernels that take one step per launch (device code): a
// workgroup of NW waves holds K * NW columns of 64 rows, one row per lane and
// column unit * NW + wave in each of a wave's K units, so that all SIMDs stay
// busy as the active columns shrink from half step to half step.  x taps come
// from LDS (four spare columns on each side, so every read stays inside), z
// taps from wave shifts; WAVE_HALO columns and rows on each side are halo.
#pragma once
#include "common.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace ds2d {

template <int K, int NW>
struct TileLanes {
    static constexpr int RX = K * NW;
    StepTile T;
    int lane, wv, z, ix0;
    bool zu, zown, zphys;
    __device__ __forceinline__ bool init(const StepTile* tiles, int ntiles, int per_xcd) {
        const int ch = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
        if (ch >= ntiles) return false;
        T = tiles[ch];
        lane = threadIdx.x & 63;
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        z = T.z0 - WAVE_HALO + lane;
        ix0 = T.x0 - WAVE_HALO;
        zu = z >= NOP && z < T.nzp - NOP;
        zown = zu && lane >= WAVE_HALO && lane < 64 - WAVE_HALO;
        zphys = z >= T.pml && z < T.pml + T.nz;
        return true;
    }
    __device__ __forceinline__ int row(int k) const { return k * NW + wv; }
    __device__ __forceinline__ int col(int k) const { return ix0 + k * NW + wv; }
    __device__ __forceinline__ bool row_upd(int k) const { return col(k) >= NOP && col(k) < T.nxp - NOP; }
    __device__ __forceinline__ bool upd(int k) const { return zu && row_upd(k); }
    __device__ __forceinline__ bool inside(int k, int m) const {
        return (k * NW >= m || row(k) >= m) && (k * NW + NW <= RX - m || row(k) < RX - m);
    }
    __device__ __forceinline__ uint32_t cell(int k) const {
        return (uint32_t)(T.off + (long long)col(k) * T.nzp + z);
    }
    __device__ __forceinline__ bool phys(int k) const { return zphys && col(k) >= T.pml && col(k) < T.pml + T.nx; }
    __device__ __forceinline__ size_t hist(int k, int it) const {
        return (size_t)T.hist_off + ((size_t)it * T.nx + (col(k) - T.pml)) * T.nz + (size_t)(z - T.pml);
    }
    __device__ __forceinline__ float dplus_x(const float* f, int k, float own) const {
        const float* X = f + (row(k) + 4) * 64 + lane;
        return taps(X[64], own, X[128], X[-64], X[192], X[-128], X[256], X[-192]);
    }
    __device__ __forceinline__ float dminus_x(const float* f, int k, float own) const {
        const float* X = f + (row(k) + 4) * 64 + lane;
        return taps(own, X[-64], X[64], X[-128], X[128], X[-192], X[192], X[-256]);
    }
    __device__ __forceinline__ bool damped(int k) const {
        return T.damp > 0 && (z < T.damp || z > T.nzp - T.damp || col(k) < T.damp || col(k) > T.nxp - T.damp);
    }
    // v with the source sample on top in the source cell
    __device__ __forceinline__ float with_source(int k, float v, float w) const {
        return col(k) == T.isx && z == T.isz ? v + w : v;
    }
    __device__ __forceinline__ void put_source(float* f, const float (&v)[K], float w) const {
#pragma unroll
        for (int k = 0; k < K; ++k) f[(row(k) + 4) * 64 + lane] = with_source(k, v[k], w);
    }
    __device__ __forceinline__ void put(float* f, const float (&v)[K]) const {
#pragma unroll
        for (int k = 0; k < K; ++k) f[(row(k) + 4) * 64 + lane] = v[k];
    }
};

}  // namespace ds2d
