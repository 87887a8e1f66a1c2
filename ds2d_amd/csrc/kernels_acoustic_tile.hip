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
// pressure).  Measured per step: 26 windows of 331x181 Born 19.3 -> 15.9 us,
// adjoint 21.1 -> 17.8, background 49 (two per-cell kernels) -> 18.6; 16 of
// 592x336 adjoint 92 (per-cell) -> 32.6, background 56 -> 31.7; one of 331x181
// 5.3 us a step.  Tiles of 48 and 64 columns have less halo but measured up to
// 40 % slower below 1 M cells and 0-10 % faster above (FP64: slower throughout);
// one wave per strip without LDS marched no faster (18.7-21 us): its halo
// columns are computed again by every strip.
#include "common.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace ds2d {

namespace {

// A tile: RX = K * NW columns of 64 rows, one wave per column at a time
// (column = unit * NW + wave); it owns all but the eight outer ones.
constexpr int NW = 8, K = ACOU_TILE_COLS / NW + 2 * WAVE_HALO / NW;
struct Tile {
    static constexpr int RX = K * NW;
    StepTile T;
    int lane, wv, z, ix0;
    bool zu, zown;
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
        return true;
    }
    __device__ __forceinline__ int row(int k) const { return k * NW + wv; }  // uniform over the wave
    __device__ __forceinline__ bool row_upd(int k) const {
        const int ix = ix0 + row(k);
        return ix >= NOP && ix < T.nxp - NOP;
    }
    __device__ __forceinline__ bool upd(int k) const { return zu && row_upd(k); }
    // whether the wave's column k is at least m columns inside the tile
    __device__ __forceinline__ bool inside(int k, int m) const {
        return (k * NW >= m || row(k) >= m) && (k * NW + NW <= RX - m || row(k) < RX - m);
    }
    __device__ __forceinline__ bool own(int k) const { return inside(k, WAVE_HALO) && row_upd(k) && zown; }
    __device__ __forceinline__ uint32_t cell(int k) const {
        return (uint32_t)(T.off + (long long)(ix0 + row(k)) * T.nzp + z);
    }
    // history cell of the window, or -1
    __device__ __forceinline__ long long hist(int k, int it) const {
        const int lx = ix0 + row(k) - T.pml, lz = z - T.pml;
        if (lx < 0 || lx >= T.nx || lz < 0 || lz >= T.nz) return -1;
        return T.hist_off + ((long long)it * T.nx + lx) * T.nz + lz;
    }
};
// x taps of the wave's column k from an LDS copy with four spare columns on
// each side: the seven other columns of a forward (backward) difference.
template <typename R>
__device__ __forceinline__ R dplus_x(const R* f, int k, int wv, int lane, R own) {
    const R* X = f + (k * NW + wv + 4) * 64 + lane;
    return taps(X[64], own, X[128], X[-64], X[192], X[-128], X[256], X[-192]);
}
template <typename R>
__device__ __forceinline__ R dminus_x(const R* f, int k, int wv, int lane, R own) {
    const R* X = f + (k * NW + wv + 4) * 64 + lane;
    return taps(own, X[-64], X[64], X[-128], X[128], X[-192], X[192], X[-256]);
}
template <typename R>
__device__ __forceinline__ void publish(R* f, int wv, int lane, const R (&v)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) f[(k * NW + wv + 4) * 64 + lane] = v[k];
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
        p[k] = vx[k] = vz[k] = bu[k] = kk[k] = src[k] = 0.f;
        if (!g.upd(k)) continue;
        const uint32_t c = g.cell(k);
        p[k] = (a.A + 2 * n)[c];
        if (g.inside(k, 4)) {
            vx[k] = a.A[c];
            vz[k] = (a.A + n)[c];
            bu[k] = a.b[c];
        }
        if (g.inside(k, 8) && g.zown) {
            kk[k] = a.k[c];
            const long long h = g.hist(k, it);
            if (h >= 0) src[k] = 2 * a.m[c] * a.hist[h];
        }
    }
    int rec = -1;  // traces of the wave's columns: lane k holds column k's
    if (a.rec && g.T.igz >= g.T.z0 && g.T.igz < g.T.z0 + WAVE_ROWS && g.lane < K) {
        const int ix = g.ix0 + g.lane * NW + g.wv;
        if (ix >= NOP && ix < g.T.nxp - NOP) rec = rmap[g.T.rmap_off + ix];
    }
    publish(lp, g.wv, g.lane, p);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 4)) continue;
        vx[k] += a.ax * bu[k] * dplus_x(lp, k, g.wv, g.lane, p[k]);
        vz[k] += a.az * bu[k] * dplus_z(p[k]);
    }
    publish(lv, g.wv, g.lane, vx);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const float dvx = dminus_x(lv, k, g.wv, g.lane, vx[k]), dvz = dminus_z(vz[k]);
        const float pn = p[k] + (kk[k] * (a.ax * dvx + a.az * dvz) + src[k]);
        if (!(g.row_upd(k) && g.zown)) continue;
        const uint32_t c = g.cell(k);
        a.B[c] = vx[k];
        (a.B + n)[c] = vz[k];
        (a.B + 2 * n)[c] = pn;
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
        lp[k] = w[k] = vx[k] = vz[k] = ux[k] = uz[k] = gr[k] = dp[k] = 0.f;
        if (!g.upd(k)) continue;
        const uint32_t c = g.cell(k);
        lp[k] = (a.A + 2 * n)[c];
        w[k] = a.k[c];
        if (g.inside(k, 4)) {
            vx[k] = a.A[c];
            vz[k] = (a.A + n)[c];
            ux[k] = a.b[c];
        }
        if (g.inside(k, 8) && g.zown) {
            const long long h = g.hist(k, it);
            if (h >= 0) {
                dp[k] = a.hist[h];
                gr[k] = a.grad[c];
            }
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
    publish(lw, g.wv, g.lane, w);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        uz[k] = ux[k];
        if (!g.inside(k, 4)) continue;
        vx[k] += -(a.ax * dplus_x(lw, k, g.wv, g.lane, w[k]));
        vz[k] += -(a.az * dplus_z(w[k]));
        ux[k] *= vx[k];  // zero outside the update region, where b was not loaded
        uz[k] *= vz[k];
    }
    publish(lu, g.wv, g.lane, ux);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const float gx = dminus_x(lu, k, g.wv, g.lane, ux[k]), gz = dminus_z(uz[k]);
        const float rk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(res), k));
        if (!(g.row_upd(k) && g.zown)) continue;
        const uint32_t c = g.cell(k);
        a.B[c] = vx[k];
        (a.B + n)[c] = vz[k];
        (a.B + 2 * n)[c] = lp[k] + -(a.ax * gx + a.az * gz) + (g.z == g.T.igz ? rk : 0.f);
        if (g.hist(k, it) >= 0) a.grad[c] = gr[k] + 2 * dp[k] * lp[k];
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
        p[k] = vx[k] = vz[k] = 0.;
        b[k] = m[k] = 0.f;
        if (!g.upd(k)) continue;
        const uint32_t c = g.cell(k);
        p[k] = (A + 2 * n)[c];
        if (g.inside(k, 4)) {
            vx[k] = A[c];
            vz[k] = (A + n)[c];
            b[k] = bu[c];
        }
        if (g.inside(k, 8)) m[k] = kk[c];
    }
    const double w = wav[it];
    const double wz = w * src_tap<double>(g.T.isz - g.z);
    publish(lp, g.wv, g.lane, p);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 4)) continue;
        double dx = dplus_x(lp, k, g.wv, g.lane, p[k]), dz = dplus_z(p[k]);
        const int d = g.T.isx - g.ix0 - g.row(k);
        if ((unsigned)(d + 3) < 8u) {
            if (g.z == g.T.isz) dx += w * src_tap<double>(d);
            if (d == 0) dz += wz;
        }
        vx[k] += ax * b[k] * dx;
        vz[k] += az * b[k] * dz;
    }
    __syncthreads();
    publish(lp, g.wv, g.lane, vx);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const double dvx = dminus_x(lp, k, g.wv, g.lane, vx[k]), dvz = dminus_z(vz[k]);
        if (!(g.row_upd(k) && g.zown)) continue;
        const double d = (double)m[k] * (ax * dvx + az * dvz);
        const uint32_t c = g.cell(k);
        B[c] = vx[k];
        (B + n)[c] = vz[k];
        (B + 2 * n)[c] = p[k] + d;
        const long long h = g.hist(k, it);
        if (h >= 0) hist[h] = (float)d;
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
