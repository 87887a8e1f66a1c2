// Plain-L2 acoustic steps of the resident-history passes (gfx950), batched
// over shot windows: Born field, adjoint, and the FP64 background that fills
// the history.  One launch per time step, one workgroup per tile.
//
// Same scheme and arithmetic as the per-cell kernels of kernels_acoustic.hip
// (the mu = 0 specialisation of born.cu:215-349 with the Born source
// 2 m dp_bg, and its transpose).
//
// A pass moves 40-60 B a cell and step, which for the batches this is used on
// comes from the Infinity Cache (a copy of such arrays runs at 7 TB/s); what
// cost more than that was the march along x, one barrier a column, with about
// one wave per SIMD to hide it.  Here a workgroup loads its tile at once
// (32 columns of 64 rows, four columns a wave), so a step is one memory
// latency, two LDS exchanges of x neighbours and wave shifts for z.  Eight
// columns and rows on each side are halo (four for the velocity, four for the
// pressure).  Measured per step: 26 windows of 331x181 Born 19.3 -> 14.2 us,
// adjoint 21.1 -> 16.4, background 49 (two per-cell kernels) -> 18.0; 16 of
// 592x336 adjoint 92 (per-cell) -> 30.2, background 56 -> 30.8; one of 331x181
// about 5 us a step.  40-58 registers and 20 KB of LDS: four workgroups a CU.  Tiles of 48 and 64 columns have less halo but measured up to
// 40 % slower below 1 M cells and 0-10 % faster above (FP64: slower throughout);
// one wave per strip without LDS marched no faster (18.7-21 us): its halo
// columns are computed again by every strip.
#include "common.hpp"
#include "kernels.hpp"
#include "tile_lanes.hpp"

namespace ds2d {

namespace {

constexpr int NW = 8, K = ACOU_TILE_COLS / NW + 2 * WAVE_HALO / NW;
using Tile = TileLanes<K, NW>;

template <typename R>
__device__ __forceinline__ void publish(R* f, const Tile& g, const R (&v)[K]) {
    g.put(f, v);
    __syncthreads();
}

}  // namespace

// Born step: v += (dt/d) b D+ p;  p += k (dt/dx D- vx + dt/dz D- vz) + 2 m dp_bg
__global__ __launch_bounds__(NW * 64) void k_acou_born_tile(AcouFusedArgs a, const StepTile* __restrict__ tiles,
                                                            int ntiles, int per_xcd, const int* __restrict__ rmap,
                                                            int nt, int it) {
    __shared__ float lp[(K * NW + 8) * 64], lv[(K * NW + 8) * 64];
    Tile g;
    if (!g.init(tiles, ntiles, per_xcd)) return;
    const long long n = a.n;
    float p[K], vx[K], vz[K], bu[K], kk[K], src[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        vx[k] = vz[k] = bu[k] = kk[k] = src[k] = 0.f;
        p[k] = g.at(a.A + 2 * n, k);
        if (g.inside(k, 4)) {
            vx[k] = g.at(a.A, k);
            vz[k] = g.at(a.A + n, k);
            bu[k] = g.at(a.b, k);
        }
        if (g.inside(k, 8)) {
            kk[k] = g.at(a.k, k);
            src[k] = 2 * g.at(a.m, k) * g.hist(a.hist, k, it);  // m is zero outside the physical window
        }
    }
    int rec = -1;  // traces of the wave's columns: lane k holds column k's
    if (a.rec && g.T.igz >= g.T.z0 && g.T.igz < g.T.z0 + WAVE_ROWS && g.lane < K) {
        const int ix = g.ix0 + g.lane * NW + g.wv;
        if (ix >= NOP && ix < g.T.nxp - NOP) rec = rmap[g.T.rmap_off + ix];
    }
    publish(lp, g, p);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 4)) continue;
        vx[k] += a.ax * bu[k] * g.dplus_x(lp, k, p[k]);
        vz[k] += a.az * bu[k] * dplus_z(p[k]);
    }
    publish(lv, g, vx);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const float dvx = g.dminus_x(lv, k, vx[k]), dvz = dminus_z(vz[k]);
        const float pn = p[k] + (kk[k] * (a.ax * dvx + a.az * dvz) + src[k]);
        if (!(g.row_upd(k) && g.zown)) continue;
        g.at(a.B, k) = vx[k];
        g.at(a.B + n, k) = vz[k];
        g.at(a.B + 2 * n, k) = pn;
        const int r = __builtin_amdgcn_readlane(rec, k);
        if (r >= 0 && g.z == g.T.igz) a.rec[g.T.rec_off + (long long)r * nt + it] = pn;
    }
}

// Adjoint step, time reversed: lp += res at the receivers;  grad += 2 dp_bg lp;
//   lv += -(dt/d) D+ (k lp);  lp += -(dt/d) D- (b lv)   (k lp, b lv masked to the update region)
// The residual of the next (earlier) step is added by the wave that stores a
// receiver's lp, as k_acou_adj_v does; the first one's by launch_acou_inj.
__global__ __launch_bounds__(NW * 64) void k_acou_adj_tile(AcouFusedArgs a, const StepTile* __restrict__ tiles,
                                                           int ntiles, int per_xcd, const int* __restrict__ rmap,
                                                           int nt, int it) {
    __shared__ float lw[(K * NW + 8) * 64], lu[(K * NW + 8) * 64];
    Tile g;
    if (!g.init(tiles, ntiles, per_xcd)) return;
    const long long n = a.n;
    float lp[K], w[K], vx[K], vz[K], ux[K], uz[K], gr[K], dp[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        vx[k] = vz[k] = ux[k] = uz[k] = gr[k] = dp[k] = 0.f;
        lp[k] = g.at(a.A + 2 * n, k);
        w[k] = g.at(a.k, k);
        if (g.inside(k, 4)) {
            vx[k] = g.at(a.A, k);
            vz[k] = g.at(a.A + n, k);
            ux[k] = g.at(a.b, k);
        }
        if (g.inside(k, 8)) {
            dp[k] = g.hist(a.hist, k, it);
            gr[k] = g.at(a.grad, k);
        }
    }
    float res = 0.f;  // residuals of the wave's columns: lane k holds column k's
    if (it > 0 && g.T.igz >= g.T.z0 && g.T.igz < g.T.z0 + WAVE_ROWS && g.lane < K) {
        const int ix = g.ix0 + g.lane * NW + g.wv;
        const int r = ix >= NOP && ix < g.T.nxp - NOP ? rmap[g.T.rmap_off + ix] : -1;
        if (r >= 0) res = a.res[g.T.rec_off + (long long)r * nt + (it - 1)];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) w[k] *= lp[k];
    publish(lw, g, w);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        uz[k] = ux[k];
        if (!g.inside(k, 4)) continue;
        vx[k] += -(a.ax * g.dplus_x(lw, k, w[k]));
        vz[k] += -(a.az * dplus_z(w[k]));
        ux[k] *= vx[k];  // zero on the frame, as b
        uz[k] *= vz[k];
    }
    publish(lu, g, ux);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const float gx = g.dminus_x(lu, k, ux[k]), gz = dminus_z(uz[k]);
        const float rk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(res), k));
        if (!(g.row_upd(k) && g.zown)) continue;
        g.at(a.B, k) = vx[k];
        g.at(a.B + n, k) = vz[k];
        g.at(a.B + 2 * n, k) = lp[k] + -(a.ax * gx + a.az * gz) + (g.z == g.T.igz ? rk : 0.f);
        if (g.phys(k)) g.at(a.grad, k) = gr[k] + 2 * dp[k] * lp[k];
    }
}

// FP64 background step A -> B (vx, vz, p) with the transient source; its
// increment, rounded once to FP32, goes to the history.
__global__ __launch_bounds__(NW * 64) void k_acou_bg_tile(const double* __restrict__ A, double* __restrict__ B,
                                                          long long n, const float* __restrict__ bu,
                                                          const float* __restrict__ kk, float* hist,
                                                          const float* __restrict__ wav,
                                                          const StepTile* __restrict__ tiles, int ntiles, int per_xcd,
                                                          double ax, double az, int it) {
    __shared__ double lp[(K * NW + 8) * 64];
    Tile g;
    if (!g.init(tiles, ntiles, per_xcd)) return;
    double p[K], vx[K], vz[K];
    float b[K], m[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        vx[k] = vz[k] = 0.;
        b[k] = m[k] = 0.f;
        p[k] = g.at(A + 2 * n, k);
        if (g.inside(k, 4)) {
            vx[k] = g.at(A, k);
            vz[k] = g.at(A + n, k);
            b[k] = g.at(bu, k);
        }
        if (g.inside(k, 8)) m[k] = g.at(kk, k);
    }
    const double w = wav[it];
    const double wz = w * src_tap<double>(g.T.isz - g.z);
    publish(lp, g, p);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 4)) continue;
        double dx = g.dplus_x(lp, k, p[k]), dz = dplus_z(p[k]);
        const int d = g.T.isx - g.ix0 - g.row(k);
        if ((unsigned)(d + 3) < 8u) {
            if (g.z == g.T.isz) dx += w * src_tap<double>(d);
            if (d == 0) dz += wz;
        }
        vx[k] += ax * b[k] * dx;
        vz[k] += az * b[k] * dz;
    }
    __syncthreads();
    publish(lp, g, vx);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const double dvx = g.dminus_x(lp, k, vx[k]), dvz = dminus_z(vz[k]);
        if (!(g.row_upd(k) && g.zown)) continue;
        const double d = (double)m[k] * (ax * dvx + az * dvz);
        g.at(B, k) = vx[k];
        g.at(B + n, k) = vz[k];
        g.at(B + 2 * n, k) = p[k] + d;
        if (g.phys(k)) g.hist(hist, k, it) = (float)d;
    }
}

void launch_acou_born_tile(hipStream_t st, const BatchShape& b, const AcouFusedArgs& a, const StepTile* tiles,
                           int ntiles, const int* rmap, int it) {
    const int per_xcd = (ntiles + 7) / 8;
    hipLaunchKernelGGL(k_acou_born_tile, dim3(per_xcd * 8), dim3(NW * 64), 0, st, a, tiles, ntiles, per_xcd, rmap,
                       b.nt, it);
}
void launch_acou_adj_tile(hipStream_t st, const BatchShape& b, const AcouFusedArgs& a, const StepTile* tiles,
                          int ntiles, const int* rmap, int it) {
    const int per_xcd = (ntiles + 7) / 8;
    hipLaunchKernelGGL(k_acou_adj_tile, dim3(per_xcd * 8), dim3(NW * 64), 0, st, a, tiles, ntiles, per_xcd, rmap,
                       b.nt, it);
}
void launch_acou_bg_tile(hipStream_t st, const BatchShape& b, const double* A, double* B, long long n, AcouMed m,
                         float* hist, const float* wav, const StepTile* tiles, int ntiles, int it) {
    const int per_xcd = (ntiles + 7) / 8;
    hipLaunchKernelGGL(k_acou_bg_tile, dim3(per_xcd * 8), dim3(NW * 64), 0, st, A, B, n, m.b, m.k, hist, wav, tiles,
                       ntiles, per_xcd, (double)b.dt / (double)b.dx, (double)b.dt / (double)b.dz, it);
}

}  // namespace ds2d
