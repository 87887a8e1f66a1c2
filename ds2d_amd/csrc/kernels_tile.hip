// Elastic forward step for batches too small to fill the chip with x-marching
// workgroups (gfx950): two time steps per launch on two-dimensional tiles,
// batched over uneven shot windows.
//
// Scheme, arithmetic, damping strips, source and recorder are those of the
// fused step (born.cu:215-349, FD2DGPU.cu:2039-2049, 355-365).
//
// What bounds a small batch is the length of a launch, not its traffic: a
// workgroup that marches 64 columns has 80 columns in series (82 us a step on
// one 141x101 padded window, 84 us on 291x141), and a launch per half step
// costs two launches (8.4-10.8 us a step).  Here every cell of a tile is loaded
// at once and a launch takes two steps, one wave per column of 64 rows: the
// state stays in registers, x neighbours come from LDS, z neighbours from the
// lanes beside (wave shifts), so a half step is one LDS exchange and about 60
// vector operations a column.  Each step spends four columns and rows on each
// side on the velocity and four on the stress, so a tile owns all but its 16
// outer ones.  Measured per launch on 291x141 with the PML: 4.4 us for the
// loads and stores alone, 9.2 us for two steps (4.6 us a step against 84 and
// 10.8); with the random boundary 7.0 us (3.5 a step).  Three steps a launch
// would leave 16 of 64 rows owned and cost more than the saved launch.
// Columns are dealt to the waves in turn (column = unit * waves + wave), which
// keeps all SIMDs busy as the active columns shrink from half step to half
// step; contiguous columns, whose x taps would partly come from registers,
// measured the same on one round and 10 % slower over several.
// Vector operations bound the PML step (1700 a wave of three columns), so the
// addresses are 32-bit offsets from scalar bases and cells beyond the update
// region rest for want of a medium instead of being masked: 10.3 -> 9.4 us from
// launch to launch on 291x141, 16 such windows 49.8 -> 45.7.  (A state that has
// overflowed reaches the frame that way a step before it would by the taps.)
// The PML tiles of 24 and 28 columns spill 36 and 44 bytes a lane at the 128 and
// 168 registers that their 14 and 12 waves leave.
#include "common.hpp"
#include "kernels.hpp"
#include "wave.hpp"

#include <type_traits>

namespace ds2d {

template <int K, int NW, bool PML>
__global__ __launch_bounds__(NW * 64) void k_tile_steps(FusedArgs a, const TileDesc* __restrict__ tiles, int ntiles,
                                                        int per_xcd, const int* __restrict__ rmap, float idx,
                                                        float idz, float dt, int nt, int it, int ns) {
    constexpr int RX = K * NW, RZ = 64, HALO = TILE_HALO;
    const int b = blockIdx.x;
    const int ch = (b % 8) * per_xcd + b / 8;
    if (ch >= ntiles) return;
    const TileDesc T = tiles[ch];
    // four spare rows on each side, so that the x taps of every row stay inside
    __shared__ float lds[4][(RX + 8) * RZ];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto row = [&](int k) { return k * NW + wv; };  // column of the tile, uniform over the wave
    auto at = [&](int f, int k) { return &lds[f][(row(k) + 4) * RZ + lane]; };
    const int z = T.z0 - HALO + lane, ix0 = T.x0 - HALO;
    const bool zu = z >= NOP && z < T.nzp - NOP;
    const bool zd = PML && T.pml > 0 && (z < T.pml || z > T.nzp - T.pml);
    const bool zown = lane >= HALO && lane < RZ - HALO && zu;
    const long long n = a.n;

    // Each component as the sum of two parts.  In a damped cell they are its x
    // and z splits, which are what its window's strips store (the sum alone with
    // one split would round the other one off at every step); elsewhere the
    // first is the component.
    float vx[K], vz[K], xx[K], zz[K], xz[K], vxb[K], vzb[K], xxb[K], zzb[K], xzb[K];
    float bx[K], lam[K], mu[K], ex[K], ez[K];
    auto row_upd = [&](int k) { const int ix = ix0 + row(k); return ix >= NOP && ix < T.nxp - NOP; };
    auto row_damp = [&](int k) { const int ix = ix0 + row(k); return T.pml > 0 && (ix < T.pml || ix > T.nxp - T.pml); };
    // Offset in bytes of column k's cell in a field, or of the nearest cell of
    // the window: those beyond it lie on its frame, which is never updated and
    // holds a resting state, so that loads need no condition.  Scalar bases and
    // 32 bits of offset (15 fields of n floats) keep 64-bit vector arithmetic,
    // which is slow, out of the addresses.
    const uint32_t nb = (uint32_t)n * 4u, zc = (uint32_t)min(max(z, 0), T.nzp - 1);
    auto cell = [&](int k) {
        return ((uint32_t)T.off + (uint32_t)min(max(ix0 + row(k), 0), T.nxp - 1) * (uint32_t)T.nzp + zc) * 4u;
    };
    auto get = [](const float* f, uint32_t o) { return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(f) + o); };
    auto set = [](float* f, uint32_t o, float v) { *reinterpret_cast<float*>(reinterpret_cast<char*>(f) + o) = v; };
    bool damped = PML && __any(zd);  // whether any cell of this wave is
#pragma unroll
    for (int k = 0; k < K; ++k) {
        vx[k] = vz[k] = xx[k] = zz[k] = xz[k] = vxb[k] = vzb[k] = xxb[k] = zzb[k] = xzb[k] = 0.f;
        bx[k] = lam[k] = mu[k] = ex[k] = ez[k] = 0.f;
        const int r = row(k);
        damped = damped || (PML && row_damp(k));
        // component f is field f of undamped cells, fields 5 + 2 f (x) and 6 + 2 f (z) of damped ones
        const uint32_t c = cell(k);
        const bool dmp = PML && (zd || row_damp(k)), u = zu && row_upd(k);  // no medium beyond u: it stays at rest
        const uint32_t step = dmp ? 2 * nb : nb, c0 = dmp ? c + 5 * nb : c, c2 = c0 + 2 * step;
        xx[k] = get(a.A, c2);
        zz[k] = get(a.A, c2 + step);
        xz[k] = get(a.A, c2 + 2 * step);
        if (dmp) {
            xxb[k] = get(a.A, c2 + nb);
            zzb[k] = get(a.A, c2 + 3 * nb);
            xzb[k] = get(a.A, c2 + 5 * nb);
        }
        if (r >= 4 && r < RX - 4) {
            vx[k] = get(a.A, c0);
            vz[k] = get(a.A, c0 + step);
            bx[k] = u ? get(a.par, c) : 0.f;
            if (dmp) {
                vxb[k] = get(a.A, c0 + nb);
                vzb[k] = get(a.A, c0 + 3 * nb);
                ex[k] = get(a.dampx, c);
                ez[k] = get(a.dampz, c);
            }
            if (r >= 8 && r < RX - 8) {
                lam[k] = u ? get(a.par, c + nb) : 0.f;
                mu[k] = u ? get(a.par, c + 2 * nb) : 0.f;
            }
        }
    }
    // traces of the wave's columns: lane k holds column k's (-1: none)
    int rec = -1;
    if (T.igz >= T.z0 && T.igz < T.z0 + RZ - 2 * HALO && lane < K) {
        const int ix = ix0 + lane * NW + wv;
        if (ix >= NOP && ix < T.nxp - NOP) rec = rmap[T.rmap_off + ix];
    }
    const float w0 = a.wav[it], w1 = ns > 1 ? a.wav[it + 1] : 0.f;
    // weight of the source in the z derivative of this lane's row
    const float cz_src = src_tap<float>(T.isz - z);
    float d1[K], r2[K], d3[K], r4[K];
    if (PML && damped) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            d1[k] = 1.f - dt * ex[k] / 2;
            r2[k] = __builtin_amdgcn_rcpf(1.f + dt * ex[k] / 2);
            d3[k] = 1.f - dt * ez[k] / 2;
            r4[k] = __builtin_amdgcn_rcpf(1.f + dt * ez[k] / 2);
        }
    }

    // One step that leaves out the MV outer columns and rows in the velocity and four more in the stress.
    auto velocity = [&](auto mvc, auto dc, float w, int step) {
        constexpr int MV = decltype(mvc)::value;
        constexpr bool DAMP = decltype(dc)::value;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int r = row(k);
            const float *X = at(0, k), *Z = at(1, k);
            float x[7], e[7];
#pragma unroll
            for (int i = 0; i < 7; ++i) {
                x[i] = X[(i < 3 ? i - 3 : i - 2) * RZ];
                e[i] = Z[(i < 4 ? i - 4 : i - 3) * RZ];
            }
            const bool all = k * NW >= MV && k * NW + NW <= RX - MV;
            if (!all && (r < MV || r >= RX - MV)) continue;
            const float txz = DAMP ? xz[k] + xzb[k] : xz[k];
            float ax = taps(x[3], DAMP ? xx[k] + xxb[k] : xx[k], x[4], x[2], x[5], x[1], x[6], x[0]);
            const float ez_ = taps(txz, e[3], e[4], e[2], e[5], e[1], e[6], e[0]);
            const float bz = dminus_z(txz);
            float cz = dplus_z(DAMP ? zz[k] + zzb[k] : zz[k]);
            // the source sample, present in this step's velocity only
            const int dx = T.isx - ix0 - r;
            if ((unsigned)(dx + 3) < 8u) {
                if (z == T.isz) ax += w * src_tap<float>(dx);
                if (dx == 0) cz += w * cz_src;
            }
            const float nx = vx[k] + bx[k] * (ax * idx + bz * idz);
            const float nz = vz[k] + bx[k] * (ez_ * idx + cz * idz);
            if (DAMP) {
                const bool d = zd || row_damp(k);
                const float ux = (d1[k] * vx[k] + bx[k] * idx * ax) * r2[k];
                const float uz = (d3[k] * vxb[k] + bx[k] * idz * bz) * r4[k];
                const float wx = (d1[k] * vz[k] + bx[k] * idx * ez_) * r2[k];
                const float wz = (d3[k] * vzb[k] + bx[k] * idz * cz) * r4[k];
                vx[k] = d ? ux : nx;
                vxb[k] = d ? uz : 0.f;
                vz[k] = d ? wx : nz;
                vzb[k] = d ? wz : 0.f;
            } else {
                vx[k] = nx;
                vz[k] = nz;
            }
            const int tr = __builtin_amdgcn_readlane(rec, k);
            if (tr >= 0 && z == T.igz && r >= HALO && r < RX - HALO) {
                const size_t o = (size_t)T.rec_off + (size_t)tr * nt + step;
                a.rec_z[o] = DAMP ? vz[k] + vzb[k] : vz[k];
                a.rec_x[o] = DAMP ? vx[k] + vxb[k] : vx[k];
            }
        }
    };
    auto stress = [&](auto msc, auto dc) {
        constexpr int MS = decltype(msc)::value;
        constexpr bool DAMP = decltype(dc)::value;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int r = row(k);
            const float *X = at(2, k), *Z = at(3, k);
            float x[7], e[7];
#pragma unroll
            for (int i = 0; i < 7; ++i) {
                x[i] = X[(i < 4 ? i - 4 : i - 3) * RZ];
                e[i] = Z[(i < 3 ? i - 3 : i - 2) * RZ];
            }
            const bool all = k * NW >= MS && k * NW + NW <= RX - MS;
            if (!all && (r < MS || r >= RX - MS)) continue;
            const float tvx = DAMP ? vx[k] + vxb[k] : vx[k], tvz = DAMP ? vz[k] + vzb[k] : vz[k];
            const float dvx = taps(tvx, x[3], x[4], x[2], x[5], x[1], x[6], x[0]) * idx;
            const float dvzx = taps(e[3], tvz, e[4], e[2], e[5], e[1], e[6], e[0]) * idx;
            const float dvz = dminus_z(tvz) * idz, dvxz = dplus_z(tvx) * idz;
            const float l = lam[k], m = mu[k], l2m = l + 2 * m;
            const float nxx = xx[k] + (l2m * dvx + l * dvz);
            const float nzz = zz[k] + (l * dvx + l2m * dvz);
            const float nxz = xz[k] + m * (dvzx + dvxz);
            if (DAMP) {
                const bool d = zd || row_damp(k);
                const float a1 = (d1[k] * xx[k] + l2m * dvx) * r2[k];
                const float a2 = (d3[k] * xxb[k] + l * dvz) * r4[k];
                const float b1 = (d1[k] * zz[k] + l * dvx) * r2[k];
                const float b2 = (d3[k] * zzb[k] + l2m * dvz) * r4[k];
                const float e1 = (d1[k] * xz[k] + m * dvzx) * r2[k];
                const float e2 = (d3[k] * xzb[k] + m * dvxz) * r4[k];
                xx[k] = d ? a1 : nxx;
                xxb[k] = d ? a2 : 0.f;
                zz[k] = d ? b1 : nzz;
                zzb[k] = d ? b2 : 0.f;
                xz[k] = d ? e1 : nxz;
                xzb[k] = d ? e2 : 0.f;
            } else {
                xx[k] = nxx;
                zz[k] = nzz;
                xz[k] = nxz;
            }
        }
    };
    auto publish = [&](int f, const float* p, const float* pb, const float* q, const float* qb) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            *at(f, k) = PML ? p[k] + pb[k] : p[k];
            *at(f + 1, k) = PML ? q[k] + qb[k] : q[k];
        }
        __syncthreads();
    };
    auto one_step = [&](auto mvc, float w, int step) {
        constexpr int MV = decltype(mvc)::value;
        publish(0, xx, xxb, xz, xzb);
        if (PML && damped)
            velocity(mvc, std::true_type{}, w, step);
        else
            velocity(mvc, std::false_type{}, w, step);
        publish(2, vx, vxb, vz, vzb);
        if (PML && damped)
            stress(std::integral_constant<int, MV + 4>{}, std::true_type{});
        else
            stress(std::integral_constant<int, MV + 4>{}, std::false_type{});
    };
    if (ns > 1) {
        one_step(std::integral_constant<int, 4>{}, w0, it);
        one_step(std::integral_constant<int, 12>{}, w1, it + 1);
    } else {
        one_step(std::integral_constant<int, 12>{}, w0, it);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int r = row(k);
        if (!zown || !row_upd(k) || r < HALO || r >= RX - HALO) continue;
        const uint32_t c = cell(k);
        if (PML && (zd || row_damp(k))) {
            const float part[10] = {vx[k], vxb[k], vz[k], vzb[k], xx[k], xxb[k], zz[k], zzb[k], xz[k], xzb[k]};
#pragma unroll
            for (int f = 0; f < 10; ++f) set(a.B, c + (5 + f) * nb, part[f]);
        } else {
            const float part[5] = {vx[k] + vxb[k], vz[k] + vzb[k], xx[k] + xxb[k], zz[k] + zzb[k], xz[k] + xzb[k]};
#pragma unroll
            for (int f = 0; f < 5; ++f) set(a.B, c + f * nb, part[f]);
        }
    }
}

void launch_tile_steps(hipStream_t st, const BatchShape& b, const FusedArgs& a, const TileDesc* tiles, int ntiles,
                       const int* rmap, int it, int ns, int kind, bool pml) {
    const int per_xcd = (ntiles + 7) / 8;
    const float idx = 1.f / b.dx, idz = 1.f / b.dz;
#define DS2D_TILE_LAUNCH(K, NW, MM)                                                                           \
    hipLaunchKernelGGL((k_tile_steps<K, NW, MM>), dim3(per_xcd * 8), dim3(NW * 64), 0, st, a, tiles, ntiles,  \
                       per_xcd, rmap, idx, idz, b.dt, b.nt, it, ns)
#define DS2D_TILE_KIND(V, K, NW)                                  \
    case V:                                                       \
        static_assert(kTiles[V].k == K && kTiles[V].nw == NW, ""); \
        if (pml)                                                  \
            DS2D_TILE_LAUNCH(K, NW, true);                        \
        else                                                      \
            DS2D_TILE_LAUNCH(K, NW, false);                       \
        break;
    switch (kind) {
        DS2D_TILE_KIND(0, 3, 14)
        DS2D_TILE_KIND(1, 4, 12)
        DS2D_TILE_KIND(2, 4, 14)
        DS2D_TILE_KIND(3, 5, 12)
    }
#undef DS2D_TILE_KIND
#undef DS2D_TILE_LAUNCH
}

}  // namespace ds2d
