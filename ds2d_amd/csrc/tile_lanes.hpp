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
    uint32_t zc, zh;  // the lane's row, inside the window and inside the physical window
    bool zu, zown, zphys;
    __device__ __forceinline__ bool init(const StepTile* tiles, int ntiles, int per_xcd) {
        const int ch = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
        if (ch >= ntiles) return false;
        T = tiles[ch];
        lane = threadIdx.x & 63;
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        z = T.z0 - WAVE_HALO + lane;
        ix0 = T.x0 - WAVE_HALO;
        zc = (uint32_t)min(max(z, 0), T.nzp - 1);
        zh = (uint32_t)min(max(z - T.pml, 0), T.nz - 1);
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
    __device__ __forceinline__ size_t hist_cell(int k, int it) const {
        return (size_t)T.hist_off + ((size_t)it * T.nx + (col(k) - T.pml)) * T.nz + (size_t)(z - T.pml);
    }
    // f at the cell of unit k, or at the nearest cell of the window: those
    // beyond it lie on its frame, which is never updated and holds a resting
    // state, so that loads need no condition.  Scalar base and column, 32 bits
    // of byte offset in the lane, so that an access costs no vector address.
    // Where issue bounds a step this pays (acoustic Born on 26 small windows
    // 15.9 -> 14.2 us, adjoint 17.8 -> 16.5); the elastic Born pair is bound by
    // memory and keeps cell (350 us against 357 on 16 large windows, and 182
    // against 237 for the adjoint, whose loads without a condition take 138
    // registers instead of 126 and so one workgroup a CU instead of two), and
    // the rotation step measured the same both ways (105 us).
    template <typename F>
    __device__ __forceinline__ F& at(F* f, int k) const {
        const uint32_t c = (uint32_t)min(max(col(k), 0), T.nxp - 1) * (uint32_t)T.nzp + zc;
        return *reinterpret_cast<F*>(reinterpret_cast<char*>(f + T.off) + c * (uint32_t)sizeof(F));
    }
    template <typename F>
    __device__ __forceinline__ const F& at(const F* f, int k) const {
        return at(const_cast<F*>(f), k);
    }
    __device__ __forceinline__ bool phys(int k) const { return zphys && col(k) >= T.pml && col(k) < T.pml + T.nx; }
    // step it of a history at the cell of unit k, or at the nearest physical cell
    __device__ __forceinline__ float& hist(float* f, int k, int it) const {
        const int lx = min(max(col(k) - T.pml, 0), T.nx - 1);
        float* p = f + T.hist_off + ((long long)it * T.nx + lx) * T.nz;
        return *reinterpret_cast<float*>(reinterpret_cast<char*>(p) + zh * 4u);
    }
    __device__ __forceinline__ const float& hist(const float* f, int k, int it) const {
        return hist(const_cast<float*>(f), k, it);
    }
    template <typename R>
    __device__ __forceinline__ R dplus_x(const R* f, int k, R own) const {
        const R* X = f + (row(k) + 4) * 64 + lane;
        return taps(X[64], own, X[128], X[-64], X[192], X[-128], X[256], X[-192]);
    }
    template <typename R>
    __device__ __forceinline__ R dminus_x(const R* f, int k, R own) const {
        const R* X = f + (row(k) + 4) * 64 + lane;
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
    template <typename R>
    __device__ __forceinline__ void put(R* f, const R (&v)[K]) const {
#pragma unroll
        for (int k = 0; k < K; ++k) f[(row(k) + 4) * 64 + lane] = v[k];
    }
};

}  // namespace ds2d
