// Kernels of the reference ELSRTM gradient (gfx950), batched over shot slots:
// two launches per forward step and three per backward step.
//
// The reference runs one kernel per operation (FD2DGPU.cu:1817-1897,
// 4700-4800): 15 launches a forward step and 13 a backward step, each 3-13 us
// on the batches it is used for, and most of them re-read what the previous
// one wrote.  Here the operations of a step that do not depend on each other
// run in one launch, one wavefield per block layer, and the Born fields
// follow the background with a lag:
//   forward launch pair k: velocity of bg(k), b(k-1), b2(k-2); then the
//     stresses of the same steps plus the Born sources bg(k) -> b, b(k-1) -> b2
//     (b's stress of step k-1 and its source of step k meet in one cell update);
//   backward step k: (1) bg stress and strain, b velocity of step k+1, bk
//     stress; (2) bg velocity, bk and bb velocity with the Born adjoint;
//     (3) b stress and source, bb stress, the images.
// Split PML memory is touched only where a damping profile can be non-zero;
// elsewhere the split update equals the unsplit one.  A field that other
// terms are added to (Born sources, Born adjoint, residuals: the next update
// drops them, because it rebuilds the sum from the splits) keeps the bare
// value of such cells in a split array and the sum in the field itself.
// The receiver side's derivatives of (moduli x stress) are taken of products
// that the stress kernel writes once per cell instead of at all 8 taps.
#include "common.hpp"
#include "kernels.hpp"

namespace ds2d {

namespace {

template <typename T>
struct Cf;
template <>
struct Cf<float> {
    static constexpr float c1 = DS2D_C1, c2 = DS2D_C2, c3 = DS2D_C3, c4 = DS2D_C4;
};
template <>
struct Cf<double> {
    static constexpr double c1 = 1225.0 / 1024.0, c2 = -245.0 / 3072.0, c3 = 49.0 / 5120.0, c4 = -5.0 / 7168.0;
};

// Forward / backward half-point differences at cell c along stride s.
template <typename T>
__device__ __forceinline__ T dp(const T* f, size_t c, int s) {
    return Cf<T>::c1 * (f[c + s] - f[c]) + Cf<T>::c2 * (f[c + 2 * s] - f[c - s]) +
           Cf<T>::c3 * (f[c + 3 * s] - f[c - 2 * s]) + Cf<T>::c4 * (f[c + 4 * s] - f[c - 3 * s]);
}
template <typename T>
__device__ __forceinline__ T dm(const T* f, size_t c, int s) {
    return Cf<T>::c1 * (f[c] - f[c - s]) + Cf<T>::c2 * (f[c + s] - f[c - 2 * s]) +
           Cf<T>::c3 * (f[c + 2 * s] - f[c - 3 * s]) + Cf<T>::c4 * (f[c + 3 * s] - f[c - 4 * s]);
}
// Weight of the cell at offset d in a forward half-point difference.
template <typename T>
__device__ __forceinline__ T tap(int d) {
    return d == 1 ? Cf<T>::c1 : d == 2 ? Cf<T>::c2 : d == 3 ? Cf<T>::c3 : d == 4 ? Cf<T>::c4 :
           d == 0 ? -Cf<T>::c1 : d == -1 ? -Cf<T>::c2 : d == -2 ? -Cf<T>::c3 : d == -3 ? -Cf<T>::c4 : T(0);
}
__device__ __forceinline__ bool damped(const SlotDesc& S, int ix, int iz) {
    return S.boundary == 0 && (ix < S.pml || ix > S.nxp - S.pml || iz < S.pml || iz > S.nzp - S.pml);
}
__device__ __forceinline__ bool interior(const SlotDesc& S, int ix, int iz) {
    return ix >= S.pml && ix < S.nxp - S.pml && iz >= S.pml && iz < S.nzp - S.pml;
}
// Place of a cell in its slot's edge bands of step it (record_edge_wavefield /
// load_edge_wavefield, FD2DGPU.cu:3674-3731: 2N cells astride each side of the
// frame), -1 outside them.  A corner cell of two bands is kept once.
__device__ __forceinline__ long long band_index(const SlotDesc& S, int ix, int iz, int it) {
    if (S.boundary != 0) return -1;
    const int N = NOP, pml = S.pml, nx = S.nx, nz = S.nz, nxp = S.nxp, nzp = S.nzp;
    const long long across = 2 * N, down = (long long)nx * across, left = 2 * down;
    const long long base = S.edge_off + (long long)it * (2 * across * nx + 2 * across * nz);
    if (ix >= pml && ix < nxp - pml) {
        if (iz >= pml - N && iz < pml + N) return base + (ix - pml) * across + (iz - (pml - N));
        if (iz >= nzp - pml - N && iz < nzp - pml + N) return base + down + (ix - pml) * across + (iz - (nzp - pml - N));
    }
    if (iz >= pml && iz < nzp - pml) {
        if (ix >= pml - N && ix < pml + N) return base + left + (long long)(ix - (pml - N)) * nz + (iz - pml);
        if (ix >= nxp - pml - N && ix < nxp - pml + N)
            return base + left + across * nz + (long long)(ix - (nxp - pml - N)) * nz + (iz - pml);
    }
    return -1;
}

// Damping factors x' = (a x + increment) * b.
template <typename T>
struct Damp {
    T d1, r2, d3, r4;
    __device__ __forceinline__ Damp(const Med& m, size_t c, T dt) {
        const T ex = dt * (T)m.dampx[c] / 2, ez = dt * (T)m.dampz[c] / 2;
        d1 = T(1) - ex;
        r2 = T(1) / (T(1) + ex);
        d3 = T(1) - ez;
        r4 = T(1) / (T(1) + ez);
    }
};

// Velocity step (born.cu:215-279): x and z parts of both increments.
template <typename T>
__device__ __forceinline__ void velocity_cell(const EFieldT<T>& f, const Med& m, const SlotDesc& S, int ix, int iz,
                                              size_t c, T dt, T dx, T dz, T w) {
    const int s = S.nzp;
    T a = dp(f.txx, c, s), cz = dp(f.tzz, c, 1);
    const T b = dm(f.txz, c, 1), e = dm(f.txz, c, s);
    // the source sample, on txx and tzz of the source cell for this update only
    if (w != T(0)) {
        if (iz == S.isz) a += w * tap<T>(S.isx - ix);
        if (ix == S.isx) cz += w * tap<T>(S.isz - iz);
    }
    const T br = T(1) / (T)m.rho[c], kx = br * (dt / dx), kz = br * (dt / dz);
    if (damped(S, ix, iz)) {
        const Damp<T> d(m, c, dt);
        const T xx = (d.d1 * f.vx_x[c] + kx * a) * d.r2, xz = (d.d3 * f.vx_z[c] + kz * b) * d.r4;
        const T zx = (d.d1 * f.vz_x[c] + kx * e) * d.r2, zz = (d.d3 * f.vz_z[c] + kz * cz) * d.r4;
        f.vx_x[c] = xx;
        f.vx_z[c] = xz;
        f.vz_x[c] = zx;
        f.vz_z[c] = zz;
        f.vx[c] = xx + xz;
        f.vz[c] = zx + zz;
    } else {
        f.vx[c] += kx * a + kz * b;
        f.vz[c] += kx * e + kz * cz;
    }
}

// Strain taps of a velocity field: dvx/dx, dvz/dz, dvx/dz, dvz/dx (unit spacing).
template <typename T>
struct Taps {
    T xx, zz, zx, xz;
    template <typename V>
    __device__ __forceinline__ Taps(const V* vx, const V* vz, size_t c, int s)
        : xx((T)dm(vx, c, s)), zz((T)dm(vz, c, 1)), zx((T)dp(vx, c, 1)), xz((T)dp(vz, c, s)) {}
};

// Born source of the velocities behind e (born.cu:351-405): added to (txx, tzz, txz).
template <typename T>
__device__ __forceinline__ void born_source(const Med& m, size_t c, T dx, T dz, const Taps<T>& e, T& xx, T& zz, T& xz) {
    const T l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu;
    const T mp = -(T)m.dmp[c], ms = -(T)m.dms[c];
    const T p = 2 * l2m * mp, q = 2 * (l2m * mp - 2 * mu * ms);
    const T ix = T(1) / dx, iz = T(1) / dz;
    xx += p * e.xx * ix + q * e.zz * iz;
    zz += q * e.xx * ix + p * e.zz * iz;
    xz += 2 * mu * ms * (e.xz * ix + e.zx * iz);
}

// Stress step (born.cu:282-349) of f when step, and the Born source of the
// field behind sv on top when sv is given.  BARE: undamped cells keep the
// stress without the source in txx_x, tzz_z, txz_x.
template <typename T, bool BARE, typename TS>
__device__ __forceinline__ void stress_cell(const EFieldT<T>& f, const Med& m, const SlotDesc& S, int ix, int iz,
                                            size_t c, T dt, T dx, T dz, bool step, const TS* svx, const TS* svz) {
    const int s = S.nzp;
    T xx, zz, xz;
    if (damped(S, ix, iz)) {
        if (!step) return;  // no source outside the physical window
        const Taps<T> e(f.vx, f.vz, c, s);
        const T l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu, kx = dt / dx, kz = dt / dz;
        const Damp<T> d(m, c, dt);
        const T a1 = (d.d1 * f.txx_x[c] + kx * l2m * e.xx) * d.r2, a2 = (d.d3 * f.txx_z[c] + kz * l * e.zz) * d.r4;
        const T b1 = (d.d1 * f.tzz_x[c] + kx * l * e.xx) * d.r2, b2 = (d.d3 * f.tzz_z[c] + kz * l2m * e.zz) * d.r4;
        const T e1 = (d.d1 * f.txz_x[c] + kx * mu * e.xz) * d.r2, e2 = (d.d3 * f.txz_z[c] + kz * mu * e.zx) * d.r4;
        f.txx_x[c] = a1;
        f.txx_z[c] = a2;
        f.tzz_x[c] = b1;
        f.tzz_z[c] = b2;
        f.txz_x[c] = e1;
        f.txz_z[c] = e2;
        f.txx[c] = a1 + a2;
        f.tzz[c] = b1 + b2;
        f.txz[c] = e1 + e2;
        return;
    }
    T *fxx = BARE ? f.txx_x : f.txx, *fzz = BARE ? f.tzz_z : f.tzz, *fxz = BARE ? f.txz_x : f.txz;
    xx = fxx[c];
    zz = fzz[c];
    xz = fxz[c];
    if (step) {
        const Taps<T> e(f.vx, f.vz, c, s);
        const T l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu, kx = dt / dx, kz = dt / dz;
        xx += kx * l2m * e.xx + kz * l * e.zz;
        zz += kx * l * e.xx + kz * l2m * e.zz;
        xz += mu * (kx * e.xz + kz * e.zx);
        fxx[c] = xx;
        fzz[c] = zz;
        fxz[c] = xz;
    }
    if (BARE) {
        if (svx && interior(S, ix, iz)) {
            const Taps<T> e(svx, svz, c, s);  // derivatives in the source field's precision
            born_source<T>(m, c, dx, dz, e, xx, zz, xz);
        }
        f.txx[c] = xx;
        f.tzz[c] = zz;
        f.txz[c] = xz;
    }
}

// Cell of a thread: 64 rows x 4 columns a block, wavefield layer = blockIdx.z % layers.
struct Where {
    int ix, iz, layer;
    size_t c;
    bool upd;
};
__device__ __forceinline__ Where where(const SlotDesc& S, int layers) {
    Where w;
    w.iz = NOP + blockIdx.x * BZ + threadIdx.x;
    w.ix = NOP + blockIdx.y * BX + threadIdx.y;
    w.layer = blockIdx.z % layers;
    w.upd = w.ix < S.nxp - NOP && w.iz < S.nzp - NOP;
    w.c = (size_t)S.off + (size_t)w.ix * S.nzp + w.iz;
    return w;
}
// vz and vx of a receiver cell into every trace that records its column.
template <typename T>
__device__ __forceinline__ void record_cell(const SlotDesc& S, const int* rmap, const int* rnext, int ix, int nt,
                                            int it, T vz, T vx, float* rz, float* rx) {
    for (int r = rmap[S.rmap_off + ix]; r >= 0; r = rnext[S.rix_off + r]) {
        const size_t o = (size_t)S.rec_off + (size_t)r * nt + it;
        rz[o] = (float)vz;
        rx[o] = (float)vx;
    }
}

}  // namespace

// Forward launch A of pair k: velocity of bg at step k, b at k-1, b2 at k-2,
// with their records and edge bands.
template <typename TB>
__global__ __launch_bounds__(256) void k_grad_fwd_v(GradFields<TB> F, Med m, GradArgs a,
                                                    const SlotDesc* __restrict__ slots, int layers, int k) {
    const SlotDesc S = slots[blockIdx.z / layers];
    const Where w = where(S, layers);
    const int it = k - w.layer;
    if (!w.upd || it < 0 || it >= a.nt) return;
    const bool rec = w.iz == S.igz;
    if (w.layer < 2) {
        const EFieldT<TB> f = w.layer == 0 ? F.bg : F.b;
        velocity_cell<TB>(f, m, S, w.ix, w.iz, w.c, (TB)a.dt, (TB)a.dx, (TB)a.dz,
                          w.layer == 0 ? (TB)a.wav[it] : TB(0));
        if (F.edges) {
            const long long e = band_index(S, w.ix, w.iz, it);
            TB* E = F.edges + (w.layer == 0 ? 0 : 2 * a.total_edge);
            if (e >= 0) {
                E[e] = f.vx[w.c];
                E[a.total_edge + e] = f.vz[w.c];
            }
        }
        if (w.layer == 1 && rec)
            record_cell(S, a.rmap, a.rnext, w.ix, a.nt, it, f.vz[w.c], f.vx[w.c], a.rs_z, a.rs_x);
    } else {
        velocity_cell<float>(F.b2, m, S, w.ix, w.iz, w.c, a.dt, a.dx, a.dz, 0.f);
        if (rec) record_cell(S, a.rmap, a.rnext, w.ix, a.nt, it, F.b2.vz[w.c], F.b2.vx[w.c], a.rs2_z, a.rs2_x);
    }
}

// Forward launch B of pair k: stress of bg at step k; of b at k-1 with the
// Born source of bg's step k on top; of b2 at k-2 with that of b's step k-1.
template <typename TB>
__global__ __launch_bounds__(256) void k_grad_fwd_s(GradFields<TB> F, Med m, GradArgs a,
                                                    const SlotDesc* __restrict__ slots, int layers, int k) {
    const SlotDesc S = slots[blockIdx.z / layers];
    const Where w = where(S, layers);
    if (!w.upd) return;
    const int it = k - w.layer;
    const bool step = it >= 0 && it < a.nt;
    const bool src = w.layer > 0 && it + 1 >= 0 && it + 1 < a.nt;
    if (!step && !src) return;
    if (w.layer == 0)
        stress_cell<TB, false, TB>(F.bg, m, S, w.ix, w.iz, w.c, (TB)a.dt, (TB)a.dx, (TB)a.dz, true, nullptr, nullptr);
    else if (w.layer == 1)
        stress_cell<TB, true, TB>(F.b, m, S, w.ix, w.iz, w.c, (TB)a.dt, (TB)a.dx, (TB)a.dz, step,
                                  src ? F.bg.vx : nullptr, F.bg.vz);
    else
        stress_cell<float, true, TB>(F.b2, m, S, w.ix, w.iz, w.c, a.dt, a.dx, a.dz, step, src ? F.b.vx : nullptr,
                                     F.b.vz);
}

// Backward launch 1 of step k: (0) bg stress one step back on the physical
// window (FD2DGPU.cu:993-1082) with its strains, from the velocities that hold
// step k's edge bands; (1) b velocity of step k+1 one step back
// (FD2DGPU.cu:903-989), then step k's edge bands; (2) receiver-side stress
// (FD2DGPU.cu:725-761, 860-895) and the products the velocities differentiate.
template <typename TB>
__global__ __launch_bounds__(256) void k_grad_bwd_1(GradFields<TB> F, Med m, GradArgs a,
                                                    const SlotDesc* __restrict__ slots, int k) {
    const SlotDesc S = slots[blockIdx.z / 3];
    const Where w = where(S, 3);
    if (!w.upd) return;
    const size_t c = w.c;
    const int s = S.nzp;
    const long long n = a.n;
    const bool in = interior(S, w.ix, w.iz);
    if (w.layer == 0) {
        if (!in) return;
        const TB dt = a.dt, dx = a.dx, dz = a.dz, kx = dt / dx, kz = dt / dz;
        const Taps<TB> e(F.lvx, F.lvz, c, s);
        const TB l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu;
        F.bg.txx[c] -= kx * l2m * e.xx + kz * l * e.zz;
        F.bg.tzz[c] -= kx * l * e.xx + kz * l2m * e.zz;
        F.bg.txz[c] -= mu * (kx * e.xz + kz * e.zx);
        a.g[c] = (float)(e.xx / dx);
        a.g[n + c] = (float)(e.zz / dz);
        a.g[2 * n + c] = (float)(e.zx / dz) + (float)(e.xz / dx);
    } else if (w.layer == 1) {
        if (k + 1 >= a.nt) return;  // the velocities are step k's already
        const long long e = F.edges ? band_index(S, w.ix, w.iz, k) : -1;
        // the bands replace the field, not the splits that the next step starts from: cells of the
        // physical window inside a band keep the bare velocity in vx_x and vz_z
        const bool held = e >= 0 && k + 2 < a.nt;
        TB vx = held ? F.b.vx_x[c] : F.b.vx[c], vz = held ? F.b.vz_z[c] : F.b.vz[c];
        if (in) {
            const TB dt = a.dt, br = TB(1) / (TB)m.rho[c], kx = br * (dt / (TB)a.dx), kz = br * (dt / (TB)a.dz);
            vx -= kx * dp(F.b.txx, c, s) + kz * dm(F.b.txz, c, 1);
            vz -= kx * dm(F.b.txz, c, s) + kz * dp(F.b.tzz, c, 1);
        }
        if (e >= 0) {
            if (in) {
                F.b.vx_x[c] = vx;
                F.b.vz_z[c] = vz;
            }
            vx = F.edges[2 * a.total_edge + e];
            vz = F.edges[3 * a.total_edge + e];
        }
        if (in || e >= 0) {
            F.b.vx[c] = vx;
            F.b.vz[c] = vz;
        }
    } else {
        const EField f = F.bk;
        const Taps<float> e(f.vx, f.vz, c, s);
        const float kx = a.dt / a.dx, kz = a.dt / a.dz;
        float xx, zz, xz;
        if (damped(S, w.ix, w.iz)) {
            const Damp<float> d(m, c, a.dt);
            xx = (d.d1 * f.txx[c] - kx * e.xx) * d.r2;
            zz = (d.d3 * f.tzz[c] - kz * e.zz) * d.r4;
            const float p = (d.d1 * f.txz_x[c] - kx * e.xz) * d.r2, q = (d.d3 * f.txz_z[c] - kz * e.zx) * d.r4;
            f.txz_x[c] = p;
            f.txz_z[c] = q;
            xz = p + q;
        } else {
            xx = f.txx[c] - kx * e.xx;
            zz = f.tzz[c] - kz * e.zz;
            xz = f.txz[c] - (kx * e.xz + kz * e.zx);
        }
        f.txx[c] = xx;
        f.tzz[c] = zz;
        f.txz[c] = xz;
        const float l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu;
        a.wk[c] = l2m * xx + l * zz;
        a.wk[n + c] = l2m * zz + l * xx;
        a.wk[2 * n + c] = mu * xz;
        const float mp = -m.dmp[c], ms = -m.dms[c];
        const float cp = 2 * l2m * mp, cx = 2 * (l2m * mp - 2 * mu * ms);
        a.pk[c] = cp * xx + cx * zz;
        a.pk[n + c] = cp * zz + cx * xx;
        a.pk[2 * n + c] = a.cs[c] * xz;
    }
}

// Receiver-side velocity (FD2DGPU.cu:591-682) from the products w; add_x and
// add_z go on top of the sum, and undamped cells that have such a term (held)
// keep the bare velocity in vx_x and vz_z.
__device__ __forceinline__ void adjoint_velocity_cell(const EField& f, const Med& m, const SlotDesc& S, int ix, int iz,
                                                      size_t c, const float* w, long long n, float dt, float dx,
                                                      float dz, bool held, float add_x, float add_z) {
    const int s = S.nzp;
    const float br = 1.f / m.rho[c], kx = br * (dt / dx), kz = br * (dt / dz);
    const float ax = kx * dp(w, c, s), az = kz * dm(w + 2 * n, c, 1);
    const float bx = kx * dm(w + 2 * n, c, s), bz = kz * dp(w + n, c, 1);
    float vx, vz;
    if (damped(S, ix, iz)) {
        const Damp<float> d(m, c, dt);
        const float xx = (d.d1 * f.vx_x[c] - ax) * d.r2, xz = (d.d3 * f.vx_z[c] - az) * d.r4;
        const float zx = (d.d1 * f.vz_x[c] - bx) * d.r2, zz = (d.d3 * f.vz_z[c] - bz) * d.r4;
        f.vx_x[c] = xx;
        f.vx_z[c] = xz;
        f.vz_x[c] = zx;
        f.vz_z[c] = zz;
        vx = xx + xz;
        vz = zx + zz;
    } else {
        vx = (held ? f.vx_x[c] : f.vx[c]) - (ax + az);
        vz = (held ? f.vz_z[c] : f.vz[c]) - (bx + bz);
        if (held) {
            f.vx_x[c] = vx;
            f.vz_z[c] = vz;
        }
    }
    f.vx[c] = vx + add_x;
    f.vz[c] = vz + add_z;
}

// Backward launch 2 of step k: (0) bg velocity one step back, and in PML
// windows the copy of it that holds step k-1's edge bands; (1) receiver-side
// velocity with the residual of step k-1 on top; (2) the receiver-side Born
// field's velocity with the Born adjoint (born.cu:408-527) on top.  txz's x
// derivative there weights both taps with the modulus of the upper one
// (born.cu:514-515), as in the reference.
template <typename TB>
__global__ __launch_bounds__(256) void k_grad_bwd_2(GradFields<TB> F, Med m, GradArgs a,
                                                    const SlotDesc* __restrict__ slots, int k) {
    const SlotDesc S = slots[blockIdx.z / 3];
    const Where w = where(S, 3);
    if (!w.upd) return;
    const size_t c = w.c;
    const int s = S.nzp;
    const long long n = a.n;
    const bool in = interior(S, w.ix, w.iz);
    if (w.layer == 0) {
        // bg itself goes on without the bands (its splits do), lv takes them
        TB vx = in ? F.bg.vx[c] : F.lvx[c], vz = in ? F.bg.vz[c] : F.lvz[c];
        if (in) {
            const TB dt = a.dt, br = TB(1) / (TB)m.rho[c], kx = br * (dt / (TB)a.dx), kz = br * (dt / (TB)a.dz);
            vx -= kx * dp(F.bg.txx, c, s) + kz * dm(F.bg.txz, c, 1);
            vz -= kx * dm(F.bg.txz, c, s) + kz * dp(F.bg.tzz, c, 1);
            F.bg.vx[c] = vx;
            F.bg.vz[c] = vz;
        }
        if (F.edges) {
            const long long e = k > 0 ? band_index(S, w.ix, w.iz, k - 1) : -1;
            if (!in) {
                // step k's bands, which the source strains of this step still see
                F.bg.vx[c] = vx;
                F.bg.vz[c] = vz;
            }
            if (e >= 0) {
                vx = F.edges[e];
                vz = F.edges[a.total_edge + e];
            }
            F.lvx[c] = vx;
            F.lvz[c] = vz;
        }
    } else if (w.layer == 1) {
        float add_x = 0.f, add_z = 0.f;
        bool held = false;
        if (w.iz == S.igz) {
            for (int r = a.rmap[S.rmap_off + w.ix]; r >= 0; r = a.rnext[S.rix_off + r]) {
                held = true;
                if (k > 0) {
                    const size_t o = (size_t)S.rec_off + (size_t)r * a.nt + (k - 1);
                    add_z += a.rs_z[o];
                    add_x += a.rs_x[o];
                }
            }
        }
        adjoint_velocity_cell(F.bk, m, S, w.ix, w.iz, c, a.wk, n, a.dt, a.dx, a.dz, held, add_x, add_z);
    } else {
        float add_x = 0.f, add_z = 0.f;
        if (in) {
            const float *cs = a.cs, *xz = F.bk.txz;
            const float odd = DS2D_C1 * (cs[c] * (xz[c] - xz[c - s])) + DS2D_C2 * (cs[c + s] * (xz[c + s] - xz[c - 2 * s])) +
                              DS2D_C3 * (cs[c + 2 * s] * (xz[c + 2 * s] - xz[c - 3 * s])) +
                              DS2D_C4 * (cs[c + 3 * s] * (xz[c + 3 * s] - xz[c - 4 * s]));
            const float br = -1.f / m.rho[c];
            add_x = br * (dp(a.pk, c, s) / a.dx + dm(a.pk + 2 * n, c, 1) / a.dz);
            add_z = br * (dp(a.pk + n, c, 1) / a.dz + odd / a.dx);
        }
        adjoint_velocity_cell(F.bb, m, S, w.ix, w.iz, c, a.wb, n, a.dt, a.dx, a.dz, in, add_x, add_z);
    }
}

// Backward launch 3 of step k: b stress one step back with its strains and
// bg's Born source on top, the receiver-side Born field's stress and products,
// and the images (FD2DGPU.cu:3235-3263, 3333-3349).
template <typename TB>
__global__ __launch_bounds__(256) void k_grad_bwd_3(GradFields<TB> F, Med m, GradArgs a,
                                                    const SlotDesc* __restrict__ slots) {
    const SlotDesc S = slots[blockIdx.z];
    const Where w = where(S, 1);
    if (!w.upd) return;
    const size_t c = w.c;
    const int s = S.nzp;
    const long long n = a.n;
    const float l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu;
    const EField f = F.bb;
    float xx, zz, xz;
    {
        const Taps<float> e(f.vx, f.vz, c, s);
        const float kx = a.dt / a.dx, kz = a.dt / a.dz;
        if (damped(S, w.ix, w.iz)) {
            const Damp<float> d(m, c, a.dt);
            xx = (d.d1 * f.txx[c] - kx * e.xx) * d.r2;
            zz = (d.d3 * f.tzz[c] - kz * e.zz) * d.r4;
            const float p = (d.d1 * f.txz_x[c] - kx * e.xz) * d.r2, q = (d.d3 * f.txz_z[c] - kz * e.zx) * d.r4;
            f.txz_x[c] = p;
            f.txz_z[c] = q;
            xz = p + q;
        } else {
            xx = f.txx[c] - kx * e.xx;
            zz = f.tzz[c] - kz * e.zz;
            xz = f.txz[c] - (kx * e.xz + kz * e.zx);
        }
        f.txx[c] = xx;
        f.tzz[c] = zz;
        f.txz[c] = xz;
        a.wb[c] = l2m * xx + l * zz;
        a.wb[n + c] = l2m * zz + l * xx;
        a.wb[2 * n + c] = mu * xz;
    }
    if (!interior(S, w.ix, w.iz)) return;
    float hxx, hzz, hxz;
    {
        const TB dt = a.dt, dx = a.dx, dz = a.dz, kx = dt / dx, kz = dt / dz;
        const TB tl = m.lam[c], tm = m.mu[c], tl2m = tl + 2 * tm;
        const Taps<TB> e(F.b.vx, F.b.vz, c, s);
        TB bxx = F.b.txx_x[c] - (kx * tl2m * e.xx + kz * tl * e.zz);
        TB bzz = F.b.tzz_z[c] - (kx * tl * e.xx + kz * tl2m * e.zz);
        TB bxz = F.b.txz_x[c] - tm * (kx * e.xz + kz * e.zx);
        F.b.txx_x[c] = bxx;
        F.b.tzz_z[c] = bzz;
        F.b.txz_x[c] = bxz;
        hxx = (float)(e.xx / dx);
        hzz = (float)(e.zz / dz);
        hxz = (float)(e.zx / dz) + (float)(e.xz / dx);
        const Taps<TB> g(F.bg.vx, F.bg.vz, c, s);
        born_source<TB>(m, c, dx, dz, g, bxx, bzz, bxz);
        F.b.txx[c] = bxx;
        F.b.tzz[c] = bzz;
        F.b.txz[c] = bxz;
    }
    const size_t o = (size_t)S.win_off + (size_t)(w.ix - S.pml) * S.nz + (w.iz - S.pml);
    const long long W = a.wstride;
    const float gxx = a.g[c], gzz = a.g[n + c], gxz = a.g[2 * n + c];
    const float kp = -2 * m.vp[c] * m.vp[c] * m.rho[c], ks = -2 * m.vs[c] * m.vs[c] * m.rho[c];
    const float axx = F.bk.txx[c], azz = F.bk.tzz[c], axz = F.bk.txz[c];
    float* w7 = a.w7;
    // background strain x receiver stress, illumination
    w7[o] += kp * ((gxx + gzz) * (axx + azz));
    w7[o + W] += ks * (-2 * (gxx * azz + gzz * axx) + gxz * axz);
    const float ux = (float)F.bg.vx[c], uz = (float)F.bg.vz[c];
    w7[o + 2 * W] += ux * ux + uz * uz;
    // scattered strain x receiver stress
    w7[o + 3 * W] += kp * ((hxx + hzz) * (axx + azz));
    w7[o + 4 * W] += ks * (-2 * (hxx * azz + hzz * axx) + hxz * axz);
    // background strain x receiver-side scattered stress
    w7[o + 5 * W] += kp * ((gxx + gzz) * (xx + zz));
    w7[o + 6 * W] += ks * (-2 * (gxx * zz + gzz * xx) + gxz * xz);
}

// Start of the backward loop: the modulus of the Born adjoint's txz, the copy
// of bg's velocity that holds the edge bands (PML windows; the last step's are
// its own values), and the last step's residual on bk's receivers (at rest).
template <typename TB>
__global__ __launch_bounds__(256) void k_grad_bwd_0(GradFields<TB> F, Med m, GradArgs a,
                                                    const SlotDesc* __restrict__ slots) {
    const SlotDesc S = slots[blockIdx.z];
    const int iz = blockIdx.x * BZ + threadIdx.x, ix = blockIdx.y * BX + threadIdx.y;
    if (ix >= S.nxp || iz >= S.nzp) return;
    const size_t c = (size_t)S.off + (size_t)ix * S.nzp + iz;
    a.cs[c] = 2 * m.mu[c] * -m.dms[c];
    if (F.lvx != F.bg.vx) {
        F.lvx[c] = F.bg.vx[c];
        F.lvz[c] = F.bg.vz[c];
    }
    if (iz == S.igz)
        for (int r = a.rmap[S.rmap_off + ix]; r >= 0; r = a.rnext[S.rix_off + r]) {
            const size_t o = (size_t)S.rec_off + (size_t)r * a.nt + (a.nt - 1);
            F.bk.vz[c] += a.rs_z[o];
            F.bk.vx[c] += a.rs_x[o];
        }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static dim3 grad_grid(const BatchShape& b, int layers) {
    return dim3(ceil_div(b.nzp - 2 * NOP, BZ), ceil_div(b.max_nxp - 2 * NOP, BX), b.nslots * layers);
}

template <typename TB>
void launch_grad_forward(hipStream_t st, const BatchShape& b, const GradFields<TB>& F, Med m, const GradArgs& a,
                         bool second) {
    const int layers = second ? 3 : 2, end = a.nt + layers - 1;
    const dim3 grid = grad_grid(b, layers), block(BZ, BX);
    for (int k = 0; k < end; ++k) {
        hipLaunchKernelGGL(k_grad_fwd_v<TB>, grid, block, 0, st, F, m, a, b.slots, layers, k);
        // the last field's last stress feeds nothing (with b2 there, b's is step nt-1's at k = nt)
        if (k + 1 < end)
            hipLaunchKernelGGL(k_grad_fwd_s<TB>, grid, block, 0, st, F, m, a, b.slots, layers, k);
    }
}

template <typename TB>
void launch_grad_backward(hipStream_t st, const BatchShape& b, const GradFields<TB>& F, Med m, const GradArgs& a) {
    const dim3 block(BZ, BX), all(ceil_div(b.nzp, BZ), ceil_div(b.max_nxp, BX), b.nslots);
    hipLaunchKernelGGL(k_grad_bwd_0<TB>, all, block, 0, st, F, m, a, b.slots);
    for (int k = a.nt - 1; k >= 0; --k) {
        hipLaunchKernelGGL(k_grad_bwd_1<TB>, grad_grid(b, 3), block, 0, st, F, m, a, b.slots, k);
        hipLaunchKernelGGL(k_grad_bwd_2<TB>, grad_grid(b, 3), block, 0, st, F, m, a, b.slots, k);
        hipLaunchKernelGGL(k_grad_bwd_3<TB>, grad_grid(b, 1), block, 0, st, F, m, a, b.slots);
    }
}

template void launch_grad_forward<float>(hipStream_t, const BatchShape&, const GradFields<float>&, Med, const GradArgs&, bool);
template void launch_grad_forward<double>(hipStream_t, const BatchShape&, const GradFields<double>&, Med, const GradArgs&, bool);
template void launch_grad_backward<float>(hipStream_t, const BatchShape&, const GradFields<float>&, Med, const GradArgs&);
template void launch_grad_backward<double>(hipStream_t, const BatchShape&, const GradFields<double>&, Med, const GradArgs&);

}  // namespace ds2d
