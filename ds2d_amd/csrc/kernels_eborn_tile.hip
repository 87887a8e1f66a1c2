// Steps of the plain-L2 elastic Born pair on tiles (gfx950), batched over shot
// windows: forward (background and scattered field, or either alone) and
// adjoint, one launch per time step.
//
// Same scheme and, contraction by contraction (eborn_math.hpp), the same
// arithmetic as the per-cell kernels of kernels_eborn.hip (born.cu:351-405 for
// the Born source, unsplit fields, random boundary): results are equal bit for
// bit.
//
// A step of the pair moves 100 B a cell (108 B backwards with the reversal),
// which bounds it on large batches; on smaller ones a march along x, with a
// barrier a column and 80 columns in series, cost 115 us a step whatever the
// size.  A workgroup of eight waves loads its tile at once, one column of 64
// rows per wave and unit, exchanges x neighbours through LDS (twice a step) and
// reads z neighbours with wave shifts; eight columns and rows on each side are
// halo.  Measured per pass: PP/PS CG on 8 windows of 592x336 with the history
// 77.8 -> 24 ms (adjoint step 116 -> 29 us, forward 118 -> 34, scattered field
// alone 25); one of 141x101 54.9 -> 5.3 ms; forward on
// 16 windows of 440-1240 x 1080 392 -> 350 us a step (4.3 TB/s of the 100 B),
// adjoint with reversal on 8 of them 208 -> 193 us.
// Width: 32 owned columns (six units, two workgroups of 126 registers a CU)
// have less halo, 16 (four units) more workgroups.  Narrow: 24.0 against 25.1 ms on
// the 8 windows (1064 wide tiles), 5.3 against 6.7 on one; wide: 56.1 against
// 59.3 ms on the 16 large windows (9900 tiles), 41.8 against 55.3 for the
// adjoint of 8 (5000).  Hence the line at 2048 wide tiles; between 1100 and
// 5000 it is not measured.  The narrow adjoint with the reversal takes 129
// registers, and so one workgroup a CU: still 22 us a step on one window of
// 592x336 and 124 on 16 against 139 and 238 with the march.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "tile_lanes.hpp"
#include "eborn_math.hpp"

namespace ds2d {

// One forward step of the background (BG) and / or the scattered field (BN).
// hist_mode 1 stores the background strains, 2 takes them from the history.
template <int K, int NW, bool BG, bool BN>
__global__ __launch_bounds__(NW * 64) void k_eb_tile(EbFusedArgs a, const StepTile* __restrict__ tiles, int ntiles,
                                                     int per_xcd, const int* __restrict__ rmap, float cax, float caz,
                                                     float idx, float idz, float w, int it, int nt, int hist_mode) {
    constexpr int NF = (BG ? 2 : 0) + (BN ? 2 : 0), FS = (K * NW + 8) * 64;
    __shared__ float lds[NF * FS];
    float *l0 = lds, *l1 = lds + FS, *l2 = lds + (BG ? 2 : 0) * FS, *l3 = l2 + FS;
    TileLanes<K, NW> g;
    if (!g.init(tiles, ntiles, per_xcd)) return;
    const long long n = a.n;
    float gvx[K], gvz[K], gxx[K], gzz[K], gxz[K], svx[K], svz[K], sxx[K], szz[K], sxz[K], br[K], lam[K], mu[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        gvx[k] = gvz[k] = gxx[k] = gzz[k] = gxz[k] = svx[k] = svz[k] = sxx[k] = szz[k] = sxz[k] = 0.f;
        br[k] = 1.f;
        lam[k] = mu[k] = 0.f;
        if (!g.upd(k)) continue;
        const uint32_t c = g.cell(k);
        if (BG) {
            gxx[k] = (a.A + 2 * n)[c];
            gxz[k] = (a.A + 4 * n)[c];
            gzz[k] = (a.A + 3 * n)[c];
        }
        if (BN) {
            sxx[k] = (a.A + 7 * n)[c];
            sxz[k] = (a.A + 9 * n)[c];
            szz[k] = (a.A + 8 * n)[c];
        }
        if (g.inside(k, 4)) {
            br[k] = a.m.rho[c];
            if (BG) {
                gvx[k] = a.A[c];
                gvz[k] = (a.A + n)[c];
            }
            if (BN) {
                svx[k] = (a.A + 5 * n)[c];
                svz[k] = (a.A + 6 * n)[c];
            }
        }
        if (g.inside(k, 8) && g.zown) {
            lam[k] = a.m.lam[c];
            mu[k] = a.m.mu[c];
        }
    }
    int rec = -1;
    if (BN && a.rec_z && g.T.igz >= g.T.z0 && g.T.igz < g.T.z0 + WAVE_ROWS && g.lane < K) {
        const int ix = g.ix0 + g.lane * NW + g.wv;
        if (ix >= NOP && ix < g.T.nxp - NOP) rec = rmap[g.T.rmap_off + ix];
    }
    if (BG) {
        g.put_source(l0, gxx, w);  // the source sample is on txx and tzz for these taps only
        g.put(l1, gxz);
    }
    if (BN) {
        g.put(l2, sxx);
        g.put(l3, sxz);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 4)) continue;
        const bool u = g.upd(k);
        const float b = 1.f / br[k];
        if (BG) {
            const float dx = g.dplus_x(l0, k, g.with_source(k, gxx[k], w)), dz = dplus_z(g.with_source(k, gzz[k], w));
            const float ex = g.dminus_x(l1, k, gxz[k]), ez = dminus_z(gxz[k]);
            gvx[k] += u ? ebm::two(b * cax, dx, b * caz, ez) : 0.f;
            gvz[k] += u ? ebm::two(b * cax, ex, b * caz, dz) : 0.f;
        }
        if (BN) {
            const float dx = g.dplus_x(l2, k, sxx[k]), dz = dplus_z(szz[k]);
            const float ex = g.dminus_x(l3, k, sxz[k]), ez = dminus_z(sxz[k]);
            svx[k] += u ? ebm::two(b * cax, dx, b * caz, ez) : 0.f;
            svz[k] += u ? ebm::two(b * cax, ex, b * caz, dz) : 0.f;
        }
    }
    __syncthreads();
    if (BG) {
        g.put(l0, gvx);
        g.put(l1, gvz);
    }
    if (BN) {
        g.put(l2, svx);
        g.put(l3, svz);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const ebm::Moduli m(lam[k], mu[k]);
        float dvx = 0.f, dvz = 0.f, dvxz = 0.f, dvzx = 0.f;
        if (BG) {
            dvx = g.dminus_x(l0, k, gvx[k]);
            dvz = dminus_z(gvz[k]);
            dvxz = dplus_z(gvx[k]);
            dvzx = g.dplus_x(l1, k, gvz[k]);
        }
        float bvx = 0.f, bvz = 0.f, bvxz = 0.f, bvzx = 0.f;
        if (BN) {
            bvx = g.dminus_x(l2, k, svx[k]);
            bvz = dminus_z(svz[k]);
            bvxz = dplus_z(svx[k]);
            bvzx = g.dplus_x(l3, k, svz[k]);
        }
        const int tr = BN ? __builtin_amdgcn_readlane(rec, k) : -1;
        if (!(g.zown && g.row_upd(k))) continue;
        const uint32_t c = g.cell(k);
        const bool phys = g.phys(k);
        float exx = dvx * idx, ezz = dvz * idz, exz = ebm::two(dvzx, idx, dvxz, idz);
        if (BG) {
            a.B[c] = gvx[k];
            (a.B + n)[c] = gvz[k];
            (a.B + 2 * n)[c] = gxx[k] + ebm::inc_xx(m, cax, caz, dvx, dvz);
            (a.B + 3 * n)[c] = gzz[k] + ebm::inc_zz(m, cax, caz, dvx, dvz);
            (a.B + 4 * n)[c] = gxz[k] + ebm::inc_xz(m, cax, caz, dvzx, dvxz);
            if (hist_mode == 1 && phys) {
                const size_t h = g.hist_cell(k, it);
                a.hist[h] = exx;
                a.hist[h + a.hstride] = ezz;
                a.hist[h + 2 * a.hstride] = exz;
            }
        }
        if (BN) {
            float txx = sxx[k] + ebm::inc_xx(m, cax, caz, bvx, bvz);
            float tzz = szz[k] + ebm::inc_zz(m, cax, caz, bvx, bvz);
            float txz = sxz[k] + ebm::inc_xz(m, cax, caz, bvzx, bvxz);
            if (phys) {
                if (!BG) {
                    const size_t h = g.hist_cell(k, it);
                    exx = a.hist[h];
                    ezz = a.hist[h + a.hstride];
                    exz = a.hist[h + 2 * a.hstride];
                }
                ebm::born_source(m, a.m.dmp[c], a.m.dms[c], exx, ezz, exz, txx, tzz, txz);
            }
            (a.B + 5 * n)[c] = svx[k];
            (a.B + 6 * n)[c] = svz[k];
            (a.B + 7 * n)[c] = txx;
            (a.B + 8 * n)[c] = tzz;
            (a.B + 9 * n)[c] = txz;
            if (tr >= 0 && g.z == g.T.igz) {
                const size_t q = (size_t)g.T.rec_off + (size_t)tr * nt + it;
                a.rec_z[q] = svz[k];
                a.rec_x[q] = svx[k];
            }
        }
    }
}

// One adjoint step (k_eb_adj_v with the residual of step it + 1, then
// k_eb_adj_s of step it).  UNDO: the background is taken one step back
// alongside; otherwise the strains come from the history.
template <int K, int NW, bool UNDO>
__global__ __launch_bounds__(NW * 64) void k_eb_adj_tile(EbAdjArgs a, const StepTile* __restrict__ tiles, int ntiles,
                                                         int per_xcd, const int* __restrict__ rmap, float cax,
                                                         float caz, float idx, float idz, float w, int it, int it_inj,
                                                         int nt) {
    constexpr int FS = (K * NW + 8) * 64;
    __shared__ float lds[(UNDO ? 4 : 2) * FS];
    float *l0 = lds, *l1 = lds + FS, *l2 = lds + (UNDO ? 2 : 0) * FS, *l3 = l2 + FS;
    TileLanes<K, NW> g;
    if (!g.init(tiles, ntiles, per_xcd)) return;
    const long long n = a.n;
    const float *Al = a.Alm, *Ag = a.Abg;
    // adjoint stress, its products C s*, velocity; background
    float xx[K], zz[K], xz[K], wa[K], wb[K], wc[K], vx[K], vz[K], br[K], lam[K], mu[K];
    float gvx[K], gvz[K], gxx[K], gzz[K], gxz[K];
    // residuals of the wave's columns: lane k holds column k's
    float rx = 0.f, rz = 0.f;
    if (it_inj >= 0 && g.T.igz >= g.T.z0 - 4 && g.T.igz < g.T.z0 + WAVE_ROWS + 4 && g.lane < K) {
        const int ix = g.ix0 + g.lane * NW + g.wv;
        const int r = ix >= NOP && ix < g.T.nxp - NOP ? rmap[g.T.rmap_off + ix] : -1;
        if (r >= 0) {
            const size_t q = (size_t)g.T.rec_off + (size_t)r * nt + it_inj;
            rx = a.res_x[q];
            rz = a.res_z[q];
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        xx[k] = zz[k] = xz[k] = vx[k] = vz[k] = br[k] = lam[k] = mu[k] = 0.f;
        gvx[k] = gvz[k] = gxx[k] = gzz[k] = gxz[k] = 0.f;
        if (!g.upd(k)) continue;
        const uint32_t c = g.cell(k);
        xx[k] = (Al + 2 * n)[c];
        zz[k] = (Al + 3 * n)[c];
        xz[k] = (Al + 4 * n)[c];
        lam[k] = a.m.lam[c];
        mu[k] = a.m.mu[c];
        if (UNDO) {
            gxx[k] = (Ag + 2 * n)[c];
            gzz[k] = (Ag + 3 * n)[c];
            gxz[k] = (Ag + 4 * n)[c];
        }
        if (g.inside(k, 4)) {
            vx[k] = Al[c];
            vz[k] = (Al + n)[c];
            br[k] = a.m.rho[c];
            if (UNDO) {
                gvx[k] = Ag[c];
                gvz[k] = (Ag + n)[c];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const ebm::Moduli m(lam[k], mu[k]);
        wa[k] = ebm::two(m.l2m, xx[k], m.l, zz[k]);
        wb[k] = ebm::two(m.l2m, zz[k], m.l, xx[k]);
        wc[k] = m.mu * xz[k];
    }
    g.put(l2, wa);
    g.put(l3, wc);
    if (UNDO) {
        g.put_source(l0, gxx, w);  // the source sample is on txx and tzz for these taps only
        g.put(l1, gxz);
    }
    __syncthreads();
    float ux[K], uz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        ux[k] = uz[k] = 0.f;
        if (!g.inside(k, 4)) continue;
        const bool u = g.upd(k);
        const float b = u ? 1.f / br[k] : 0.f;
        if (UNDO) {
            const float dx = g.dplus_x(l0, k, g.with_source(k, gxx[k], w)), dz = dplus_z(g.with_source(k, gzz[k], w));
            const float ex = g.dminus_x(l1, k, gxz[k]), ez = dminus_z(gxz[k]);
            gvx[k] -= ebm::two(b * cax, dx, b * caz, ez);
            gvz[k] -= ebm::two(b * cax, ex, b * caz, dz);
        }
        const float dx = g.dplus_x(l2, k, wa[k]), dz = dplus_z(wb[k]);
        const float ex = g.dminus_x(l3, k, wc[k]), ez = dminus_z(wc[k]);
        const float qx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rx), k));
        const float qz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rz), k));
        const bool at = g.z == g.T.igz;
        vx[k] = vx[k] + (at ? qx : 0.f) - ebm::two(cax, dx, caz, ez);
        vz[k] = vz[k] + (at ? qz : 0.f) - ebm::two(caz, dz, cax, ex);
        ux[k] = b * vx[k];
        uz[k] = b * vz[k];
    }
    __syncthreads();
    g.put(l2, ux);
    g.put(l3, uz);
    if (UNDO) {
        g.put(l0, gvx);
        g.put(l1, gvz);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!g.inside(k, 8)) continue;
        const float dxx = g.dminus_x(l2, k, ux[k]), dzz = dminus_z(uz[k]);
        const float dxz = g.dplus_x(l3, k, uz[k]), dzx = dplus_z(ux[k]);
        float dvx = 0.f, dvz = 0.f, dvxz = 0.f, dvzx = 0.f;
        if (UNDO) {
            dvx = g.dminus_x(l0, k, gvx[k]);
            dvz = dminus_z(gvz[k]);
            dvxz = dplus_z(gvx[k]);
            dvzx = g.dplus_x(l1, k, gvz[k]);
        }
        if (!(g.zown && g.row_upd(k))) continue;
        const uint32_t c = g.cell(k);
        const float txx = ebm::fma_(-cax, dxx, xx[k]), tzz = ebm::fma_(-caz, dzz, zz[k]);
        const float txz = xz[k] - ebm::two(caz, dzx, cax, dxz);
        const ebm::Moduli m(lam[k], mu[k]);
        a.Blm[c] = vx[k];
        (a.Blm + n)[c] = vz[k];
        (a.Blm + 2 * n)[c] = txx;
        (a.Blm + 3 * n)[c] = tzz;
        (a.Blm + 4 * n)[c] = txz;
        const bool phys = g.phys(k);
        float exx = dvx * idx, ezz = dvz * idz, exz = ebm::two(dvzx, idx, dvxz, idz);
        if (UNDO) {
            a.Bbg[c] = gvx[k];
            (a.Bbg + n)[c] = gvz[k];
            (a.Bbg + 2 * n)[c] = gxx[k] - ebm::inc_xx(m, cax, caz, dvx, dvz);
            (a.Bbg + 3 * n)[c] = gzz[k] - ebm::inc_zz(m, cax, caz, dvx, dvz);
            (a.Bbg + 4 * n)[c] = gxz[k] - ebm::inc_xz(m, cax, caz, dvzx, dvxz);
        } else if (phys) {
            const size_t h = g.hist_cell(k, it);
            exx = a.hist[h];
            ezz = a.hist[h + a.hstride];
            exz = a.hist[h + 2 * a.hstride];
        }
        if (phys) {
            float pp = a.gpp[c], ps = a.gps[c];
            ebm::image(m, exx, ezz, exz, txx, tzz, txz, pp, ps);
            a.gpp[c] = pp;
            a.gps[c] = ps;
        }
    }
}

static constexpr int kNW = 8;  // waves of a workgroup, and so columns per unit

StepTiles plan_step_tiles(const std::vector<int>& nxp, int nzp, int narrow, int wide) {
    long long t = 0;
    for (int w : nxp)
        t += (long long)ceil_div(std::max(w - 2 * NOP, 0), wide) * ceil_div(std::max(nzp - 2 * NOP, 0), WAVE_ROWS);
    return t >= 2048 ? StepTiles{true, wide} : StepTiles{false, narrow};
}

StepTiles plan_eb_tiles(const std::vector<int>& nxp, int nzp) {
    return plan_step_tiles(nxp, nzp, 4 * kNW - 2 * WAVE_HALO, 6 * kNW - 2 * WAVE_HALO);
}

void launch_eb_tile(hipStream_t st, const BatchShape& b, const EbFusedArgs& a, const StepTile* tiles, int ntiles,
                    bool wide, const int* rmap, float w, int it, bool do_bg, bool do_bn, int hist_mode) {
    const int per_xcd = (ntiles + 7) / 8;
    const float cax = b.dt / b.dx, caz = b.dt / b.dz, idx = 1.f / b.dx, idz = 1.f / b.dz;
#define DS2D_EB_LAUNCH(K, G, N)                                                                                    \
    hipLaunchKernelGGL((k_eb_tile<K, kNW, G, N>), dim3(per_xcd * 8), dim3(kNW * 64), 0, st, a, tiles, ntiles,      \
                       per_xcd, rmap, cax, caz, idx, idz, w, it, b.nt, hist_mode)
#define DS2D_EB_FIELDS(K)                        \
    if (do_bg && do_bn)                          \
        DS2D_EB_LAUNCH(K, true, true);           \
    else if (do_bg)                              \
        DS2D_EB_LAUNCH(K, true, false);          \
    else                                         \
        DS2D_EB_LAUNCH(K, false, true);
    if (wide) {
        DS2D_EB_FIELDS(6)
    } else {
        DS2D_EB_FIELDS(4)
    }
#undef DS2D_EB_FIELDS
#undef DS2D_EB_LAUNCH
}

void launch_eb_adj_tile(hipStream_t st, const BatchShape& b, const EbAdjArgs& a, const StepTile* tiles, int ntiles,
                        bool wide, const int* rmap, float w, int it, int it_inj, bool undo) {
    const int per_xcd = (ntiles + 7) / 8;
    const float cax = b.dt / b.dx, caz = b.dt / b.dz, idx = 1.f / b.dx, idz = 1.f / b.dz;
#define DS2D_EBA_LAUNCH(K, U)                                                                                   \
    hipLaunchKernelGGL((k_eb_adj_tile<K, kNW, U>), dim3(per_xcd * 8), dim3(kNW * 64), 0, st, a, tiles, ntiles,  \
                       per_xcd, rmap, cax, caz, idx, idz, w, it, it_inj, b.nt)
    if (wide && undo)
        DS2D_EBA_LAUNCH(6, true);
    else if (wide)
        DS2D_EBA_LAUNCH(6, false);
    else if (undo)
        DS2D_EBA_LAUNCH(4, true);
    else
        DS2D_EBA_LAUNCH(4, false);
#undef DS2D_EBA_LAUNCH
}

}  // namespace ds2d
