// One time step of the P/S-decoupled (theta/omega rotation) scheme in a
// single launch for gfx950, batched over shot windows: the velocity from the
// theta / omega gradients (GPUcalculate_rotation_v, FD2DGPU.cu:3005-3040)
// and theta / omega from the new velocity (GPUcalculate_rotation_p,
// FD2DGPU.cu:3042-3080), with the source sample on theta for this step's
// velocity update (FD2DGPU.cu:2046-2049, 1407) and the recorder of vz, vx.
//
// State per cell: theta, omega, vx, vz and, in the damping strips, the x split
// of theta and omega (the other split is the total minus it).  The P and S
// parts of a velocity component share its damping factor, so their sum takes
// the same step and is all that theta, omega and the records need; outside the
// strips the split update equals the unsplit one.
//
// 6 floats in and 4 out per cell and step bound it on large batches: 40 B (24
// more in the strips), against 56 B with the four velocity parts kept apart and
// 120 B for k_rot_v + k_rot_p.  On tiles (tile_lanes.hpp) the next bound is the
// issue of vector operations, 280 per 64 owned cells with the halo.  Measured
// on 16 windows of 440-1240 x 640: 105 us a step (344 MB of fields, 73 us at
// the rate of a large copy), against 196 us for a march along x with LDS
// columns; one 141x101 window 8.6 us against 84.  Errors against 64 bits fall
// from 5.4e-7 to 4.8e-7 with the fewer sums.
// Width: 48 owned columns (eight units, less halo) take 23.3 ms against 24.2
// of 16 (four units, two workgroups a CU and more of them) on those 16 windows
// (4200 wide tiles), 8.4 against 6.9 on 16 of 592x336 (1456) and 4.8 against
// 3.5 on one of 141x101; five or six units and 12 or 16 waves lie between.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "tile_lanes.hpp"

namespace ds2d {

template <int K, int NW, bool PML>
__global__ __launch_bounds__(NW * 64) void k_rot_tile(RotFusedArgs a, const StepTile* __restrict__ tiles, int ntiles,
                                                      int per_xcd, const int* __restrict__ rmap, float dt, float rx,
                                                      float rz, int nt, int it) {
    constexpr int FS = (K * NW + 8) * 64;
    __shared__ float lds[4 * FS];
    float *l0 = lds, *l1 = lds + FS, *l2 = lds + 2 * FS, *l3 = lds + 3 * FS;
    TileLanes<K, NW> g;
    if (!g.init(tiles, ntiles, per_xcd)) return;
    const long long n = a.n;
    float th[K], om[K], vx[K], vz[K], p2[K], s2[K], ex[K], ez[K], thx[K], omx[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        th[k] = om[k] = vx[k] = vz[k] = p2[k] = s2[k] = ex[k] = ez[k] = thx[k] = omx[k] = 0.f;
        if (!g.upd(k)) continue;
        const uint32_t c = g.cell(k);
        th[k] = a.A[c];
        om[k] = (a.A + n)[c];
        if (!g.inside(k, 4)) continue;
        vx[k] = (a.A + 2 * n)[c];
        vz[k] = (a.A + 3 * n)[c];
        p2[k] = a.vp[c];
        s2[k] = a.vs[c];
        if (PML && g.damped(k)) {
            ex[k] = a.dampx[c];
            ez[k] = a.dampz[c];
            if (g.inside(k, 8) && g.zown) {
                thx[k] = (a.A + 4 * n)[c];
                omx[k] = (a.A + 5 * n)[c];
            }
        }
    }
    int rec = -1;  // traces of the wave's columns: lane k holds column k's
    if (g.T.igz >= g.T.z0 && g.T.igz < g.T.z0 + WAVE_ROWS && g.lane < K) {
        const int ix = g.ix0 + g.lane * NW + g.wv;
        if (ix >= NOP && ix < g.T.nxp - NOP) rec = rmap[g.T.rmap_off + ix];
    }
    const float w = a.wav[it];
    g.put_source(l0, th, w);  // the source sample is on theta for these taps only
    g.put(l1, om);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 4)) continue;
        const float ts = g.with_source(k, th[k], w);
        const float tx = g.dminus_x(l0, k, ts), tz = dminus_z(ts);
        const float ox = g.dplus_x(l1, k, om[k]), oz = dplus_z(om[k]);
        const float p = p2[k] * p2[k], s = s2[k] * s2[k];
        const float dvx = p * rx * tx + s * rz * oz, dvz = p * rz * tz - s * rx * ox;
        float nvx = vx[k] + dvx, nvz = vz[k] + dvz;
        if (PML && __any(g.damped(k))) {
            const float hx = dt * ex[k] / 2, hz = dt * ez[k] / 2;  // 0 outside the strips
            nvx = ((1.f - hx) * vx[k] + dvx) / (1.f + hx);
            nvz = ((1.f - hz) * vz[k] + dvz) / (1.f + hz);
        }
        const bool u = g.upd(k);
        vx[k] = u ? nvx : 0.f;
        vz[k] = u ? nvz : 0.f;
        const int tr = __builtin_amdgcn_readlane(rec, k);
        if (tr >= 0 && g.inside(k, 8) && g.zown && g.z == g.T.igz) {
            const size_t q = (size_t)g.T.rec_off + (size_t)tr * nt + it;
            a.rec_z[q] = vz[k];
            a.rec_x[q] = vx[k];
        }
    }
    g.put(l2, vx);
    g.put(l3, vz);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const float xx = g.dplus_x(l2, k, vx[k]), xz = dminus_z(vx[k]);
        const float zx = g.dminus_x(l3, k, vz[k]), zz = dplus_z(vz[k]);
        if (!(g.zown && g.row_upd(k))) continue;
        const uint32_t c = g.cell(k);
        float t = th[k] + (rx * xx + rz * zz), o = om[k] + (rz * xz - rx * zx);
        if (PML && g.damped(k)) {
            const float hx = dt * ex[k] / 2, hz = dt * ez[k] / 2;
            const float r2 = 1.f / (1.f + hx), r4 = 1.f / (1.f + hz);
            const float tx = ((1.f - hx) * thx[k] + rx * xx) * r2, ox = ((1.f - hx) * omx[k] - rx * zx) * r2;
            t = tx + ((1.f - hz) * (th[k] - thx[k]) + rz * zz) * r4;
            o = ox + ((1.f - hz) * (om[k] - omx[k]) + rz * xz) * r4;
            (a.B + 4 * n)[c] = tx;
            (a.B + 5 * n)[c] = ox;
        }
        a.B[c] = t;
        (a.B + n)[c] = o;
        (a.B + 2 * n)[c] = vx[k];
        (a.B + 3 * n)[c] = vz[k];
    }
}

static constexpr int kNW = 8;  // waves of a workgroup, and so columns per unit

StepTiles plan_rot_tiles(const std::vector<int>& nxp, int nzp) {
    return plan_step_tiles(nxp, nzp, 4 * kNW - 2 * WAVE_HALO, 8 * kNW - 2 * WAVE_HALO);
}

void launch_rot_tile(hipStream_t st, const BatchShape& b, const RotFusedArgs& a, const StepTile* tiles, int ntiles,
                     bool wide, const int* rmap, int it, bool pml) {
    const int per_xcd = (ntiles + 7) / 8;
#define DS2D_ROT_LAUNCH(K, M)                                                                                \
    hipLaunchKernelGGL((k_rot_tile<K, kNW, M>), dim3(per_xcd * 8), dim3(kNW * 64), 0, st, a, tiles, ntiles, \
                       per_xcd, rmap, b.dt, b.dt / b.dx, b.dt / b.dz, b.nt, it)
    if (wide && pml)
        DS2D_ROT_LAUNCH(8, true);
    else if (wide)
        DS2D_ROT_LAUNCH(8, false);
    else if (pml)
        DS2D_ROT_LAUNCH(4, true);
    else
        DS2D_ROT_LAUNCH(4, false);
#undef DS2D_ROT_LAUNCH
}

}  // namespace ds2d
