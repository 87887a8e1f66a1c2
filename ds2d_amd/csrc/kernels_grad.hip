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
// value of such cells in a split array and the sum in the field itself.  The
// receiver side's
// undamped sums of FP32 keep what they round off in a split array and take it
// along in the next step (compensated summation): as one plain total instead of
// two splits they were 5-6 % further from 64 bits in the images of the
// receiver-side Born field (12 inputs each of 8 windows of 291x141 and one of
// 141x101), so they are 4-7 % nearer than two splits, for 0.5 % of the time.
// The receiver side's derivatives of (moduli x stress) are taken of products
// that the stress kernel writes once per cell instead of at all 8 taps.
//
// A launch moves 40-95 MB on 8 windows of 291x141 with the PML (6-14 us at the
// rate of cached arrays) and issues 3-5 million vector operations (6-9 us); what
// bounds it is how well the two overlap, and below 3 windows its length.  One
// cell a thread with all eight taps from memory (35 loads a cell and field) took
// 20.6-37.5 us a launch there, 126 a step of both loops.  Here a wave holds a
// column of 64 rows, loads every operand once and ahead, and takes x taps from
// LDS and z taps by wave shifts; columns are addressed by 32-bit offsets from
// scalar bases, and neighbouring tiles share an XCD's L2: 16.6-27.2 us, 99 a
// step.  8 shots x 700 steps 89.7 -> 70.4 ms (148 with a launch per operation),
// one 141x101 window x 400 steps 11.0 -> 10.1, 26 shots x 100 steps 34.  Two
// columns a wave lose more to occupancy (76 ms) than they save in halo columns,
// 16 waves to a workgroup likewise (81 ms); all fields of a launch in one
// workgroup, sharing strains, 93 ms (145-227 VGPRs, one workgroup a CU).
#include "common.hpp"
#include "kernels.hpp"
#include "slot_address.hpp"
#include "wave.hpp"

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

// dt/dx, dt/dz, 1/dx, 1/dz
template <typename T>
struct Ratios {
    T kx, kz, ix, iz;
};
template <typename T>
__device__ __forceinline__ Ratios<T> ratios(const GradArgs& a) {
    if constexpr (sizeof(T) == 8)
        return {a.kx64, a.kz64, a.ix64, a.iz64};
    else
        return {a.kx, a.kz, a.ix, a.iz};
}

template <typename T>
__device__ __forceinline__ T eight(T a1, T b1, T a2, T b2, T a3, T b3, T a4, T b4) {
    return Cf<T>::c1 * (a1 - b1) + Cf<T>::c2 * (a2 - b2) + Cf<T>::c3 * (a3 - b3) + Cf<T>::c4 * (a4 - b4);
}
// Forward / backward half-point differences along z (wave shifts: all lanes take part).
template <typename T>
__device__ __forceinline__ T zp(T f) {
    const T p1 = next_z(f), p2 = next_z(p1), p3 = next_z(p2), p4 = next_z(p3);
    const T m1 = prev_z(f), m2 = prev_z(m1), m3 = prev_z(m2);
    return eight(p1, f, p2, m1, p3, m2, p4, m3);
}
template <typename T>
__device__ __forceinline__ T zm(T f) {
    const T p1 = next_z(f), p2 = next_z(p1), p3 = next_z(p2);
    const T m1 = prev_z(f), m2 = prev_z(m1), m3 = prev_z(m2), m4 = prev_z(m3);
    return eight(f, m1, p1, m2, p2, m3, p3, m4);
}
// The same along x at a column of a tile in LDS (64 rows to a column).
template <typename T>
__device__ __forceinline__ T xp(const T* X) {
    return eight(X[64], X[0], X[128], X[-64], X[192], X[-128], X[256], X[-192]);
}
template <typename T>
__device__ __forceinline__ T xm(const T* X) {
    return eight(X[0], X[-64], X[64], X[-128], X[128], X[-192], X[192], X[-256]);
}
// Weight of the cell at offset d in a forward half-point difference.
template <typename T>
__device__ __forceinline__ T tap(int d) {
    return d == 1 ? Cf<T>::c1 : d == 2 ? Cf<T>::c2 : d == 3 ? Cf<T>::c3 : d == 4 ? Cf<T>::c4 :
           d == 0 ? -Cf<T>::c1 : d == -1 ? -Cf<T>::c2 : d == -2 ? -Cf<T>::c3 : d == -3 ? -Cf<T>::c4 : T(0);
}

// A workgroup's tile: a wave per column, eight columns, 64 rows of which the
// outer four on each side are halo.  Each wave also loads one of the four halo
// columns on each side.
constexpr int GROWS = 64 - 2 * NOP;
struct GradGrid {
    int zt, xt, layers, total, per_xcd;
};
struct GradTile {
    static constexpr int COLS = 8, FS = (COLS + 2 * NOP) * 64;
    SlotDesc S;
    int lane, wv, x0, z, layer;
    long long start, halo_start;  // of the wave's own and halo column
    bool zin, zupd;
    // Tile of this workgroup among zt x xt of each slot and layer; each XCD
    // (workgroups go round them) takes one range of them, so that the halo it
    // shares is fetched into one L2.
    __device__ __forceinline__ bool init(const SlotDesc* slots, GradGrid t) {
        int i = (blockIdx.x % 8) * t.per_xcd + blockIdx.x / 8;
        if (i >= t.total) return false;
        const int zi = i % t.zt;
        i /= t.zt;
        const int xi = i % t.xt;
        i /= t.xt;
        layer = i % t.layers;
        S = slots[i / t.layers];
        x0 = NOP + xi * COLS;
        lane = threadIdx.x & 63;
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        z = zi * GROWS + lane;
        zin = z < S.nzp;
        zupd = lane >= NOP && lane < 64 - NOP && z < S.nzp - NOP;
        start = uniform(column_start(S.off, col(), S.nzp));
        halo_start = uniform(column_start(S.off, halo_col(), S.nzp));
        return x0 < S.nxp - NOP;
    }
    // kept in scalar registers: else the compiler adds a lane's offset to it first, in 64-bit vector arithmetic
    static __device__ __forceinline__ long long uniform(long long v) {
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
        return (long long)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32)) << 32 | lo);
    }
    __device__ __forceinline__ int col() const { return x0 + wv; }
    __device__ __forceinline__ int halo_col() const { return wv < NOP ? x0 - NOP + wv : x0 + COLS + wv - NOP; }
    __device__ __forceinline__ bool own() const { return col() < S.nxp - NOP; }
    // f at the lane's cell
    template <typename T>
    __device__ __forceinline__ T& at(T* f) const {
        return column_cell(f, start, z);
    }
    // the lane's cell in an image window
    __device__ __forceinline__ float& window(float* w) const {
        return column_cell(w, column_start(S.win_off, col() - S.pml, S.nz), z - S.pml);
    }
    __device__ __forceinline__ int place() const { return (wv + NOP) * 64 + lane; }
    // One mask each, without branches, and what a cell's kind decides is a
    // value and not an address: of loads of one register in both arms of an if
    // behind such a chain of conditions the compiler (ROCm 7.2) made one load of
    // a selected address, and lost the choice of the lanes above and below the
    // physical window. So the total is loaded by every cell of the region and
    // replaced where the state is another one.
    __device__ __forceinline__ bool upd() const { return zupd & own(); }
    __device__ __forceinline__ bool interior() const {
        return (col() >= S.pml) & (col() < S.nxp - S.pml) & (z >= S.pml) & (z < S.nzp - S.pml);
    }
    __device__ __forceinline__ bool damped() const {
        return (S.boundary == 0) & ((col() < S.pml) | (col() > S.nxp - S.pml) | (z < S.pml) | (z > S.nzp - S.pml));
    }
    // values of the wave's own column, of its halo column
    template <typename T>
    __device__ __forceinline__ void load(const T* f, T& r) const {
        r = zin && col() < S.nxp ? at(f) : T(0);
    }
    template <typename T>
    __device__ __forceinline__ T halo(const T* f) const {
        return zin && halo_col() < S.nxp ? column_cell(f, halo_start, z) : T(0);
    }
    template <typename T>
    __device__ __forceinline__ void put(T* lds, const T& r, T h) const {
        lds[place()] = r;
        lds[(wv < NOP ? wv : COLS + wv) * 64 + lane] = h;
    }
};

constexpr int GTHREADS = GradTile::COLS * 64;

// Samples of a slot's edge bands a step.
__device__ __forceinline__ long long band_step(const SlotDesc& S) { return 4 * NOP * (S.nx + S.nz); }
// Place of a cell in its slot's edge bands of a step (record_edge_wavefield /
// load_edge_wavefield, FD2DGPU.cu:3674-3731: 2N cells astride each side of the
// frame), -1 outside them.  A corner cell of two bands is kept once.
__device__ __forceinline__ int band_place(const SlotDesc& S, int ix, int iz) {
    const int N = NOP, pml = S.pml, across = 2 * N, down = S.nx * across, left = 2 * down;
    const int ex = S.nxp - pml, ez = S.nzp - pml;
    int r = -1;
    if (S.boundary != 0) return r;
    if (ix >= pml && ix < ex) {
        if (iz >= pml - N && iz < pml + N) r = (ix - pml) * across + iz - (pml - N);
        else if (iz >= ez - N && iz < ez + N) r = down + (ix - pml) * across + iz - (ez - N);
    }
    if (r < 0 && iz >= pml && iz < ez) {
        if (ix >= pml - N && ix < pml + N) r = left + (ix - (pml - N)) * S.nz + iz - pml;
        else if (ix >= ex - N && ix < ex + N) r = left + across * S.nz + (ix - (ex - N)) * S.nz + iz - pml;
    }
    return r;
}

// Damping factors x' = (a x + increment) * b.
template <typename T>
struct Damp {
    T d1, r2, d3, r4;
    __device__ __forceinline__ Damp(float dampx, float dampz, T dt) {
        const T ex = dt * (T)dampx / 2, ez = dt * (T)dampz / 2;
        d1 = T(1) - ex;
        r2 = T(1) / (T(1) + ex);
        d3 = T(1) - ez;
        r4 = T(1) / (T(1) + ez);
    }
};
// Damping of the damped cells, loaded ahead.
struct DampState {
    float x, z;
    __device__ __forceinline__ void load(const GradTile& g, const Med& m) {
        x = z = 0.f;
        if (g.upd() && g.damped()) {
            x = g.at(m.dampx);
            z = g.at(m.dampz);
        }
    }
};
// A medium array at the updated cells, loaded ahead.
struct MedState {
    float v;
    __device__ __forceinline__ void load(const GradTile& g, const float* f) {
        v = g.upd() ? g.at(f) : 1.f;
    }
};

// Stress of a wavefield whose derivatives the velocity takes: own columns and
// the halo column of the two x-differentiated components.
template <typename T>
struct Stress3 {
    T xx, zz, xz, hxx, hxz;
    __device__ __forceinline__ void load(const GradTile& g, const T* fxx, const T* fzz, const T* fxz) {
        g.load(fxx, xx);
        g.load(fzz, zz);
        g.load(fxz, xz);
        hxx = g.halo(fxx);
        hxz = g.halo(fxz);
    }
    __device__ __forceinline__ void put(const GradTile& g, T* l) const {
        g.put(l, xx, hxx);
        g.put(l + GradTile::FS, xz, hxz);
    }
};
// The four differences of a stress: dxx/dx, dxz/dz, dxz/dx, dzz/dz.
template <typename T>
struct Grad4 {
    T a, b, e, d;
    __device__ __forceinline__ Grad4(const GradTile& g, const Stress3<T>& s, const T* l)
        : a(xp(l + g.place())), b(zm(s.xz)), e(xm(l + GradTile::FS + g.place())), d(zp(s.zz)) {}
};

// Velocity of a wavefield, whose strains the stress takes.
template <typename T>
struct Vel2 {
    T vx, vz, hx, hz;
    __device__ __forceinline__ void load(const GradTile& g, const T* x, const T* z) {
        g.load(x, vx);
        g.load(z, vz);
        hx = g.halo(x);
        hz = g.halo(z);
    }
    __device__ __forceinline__ void put(const GradTile& g, T* l) const {
        g.put(l, vx, hx);
        g.put(l + GradTile::FS, vz, hz);
    }
};
// Strain taps: dvx/dx, dvz/dz, dvx/dz, dvz/dx (unit spacing).
template <typename T>
struct Taps {
    T xx, zz, zx, xz;
    __device__ __forceinline__ Taps(const GradTile& g, const Vel2<T>& v, const T* l)
        : xx(xm(l + g.place())), zz(zm(v.vz)), zx(zp(v.vx)), xz(xp(l + GradTile::FS + g.place())) {}
    template <typename U>
    __device__ __forceinline__ explicit Taps(const Taps<U>& u) : xx((T)u.xx), zz((T)u.zz), zx((T)u.zx), xz((T)u.xz) {}
};

// State of a velocity update, loaded ahead of the derivatives: the splits of
// damped cells, the components of the others.
template <typename T>
struct VelState {
    T p, q, pz, qz;
    __device__ __forceinline__ void load(const GradTile& g, const EFieldT<T>& f) {
        p = q = pz = qz = T(0);
        if (!g.upd()) return;
        p = g.at(f.vx);
        q = g.at(f.vz);
        if (g.damped()) {
            p = g.at(f.vx_x);
            q = g.at(f.vz_x);
            pz = g.at(f.vx_z);
            qz = g.at(f.vz_z);
        }
    }
};
// Velocity step (born.cu:215-279) of an updated cell; vx and vz are its results.
template <typename T>
__device__ __forceinline__ void velocity_cell(const GradTile& g, const EFieldT<T>& f, const VelState<T>& v,
                                              const DampState& ds, T dt, T kx, T kz, const Grad4<T>& t, T& vx,
                                              T& vz) {
    if (g.damped()) {
        const Damp<T> d(ds.x, ds.z, dt);
        const T xx = (d.d1 * v.p + kx * t.a) * d.r2, xz = (d.d3 * v.pz + kz * t.b) * d.r4;
        const T zx = (d.d1 * v.q + kx * t.e) * d.r2, zz = (d.d3 * v.qz + kz * t.d) * d.r4;
        g.at(f.vx_x) = xx;
        g.at(f.vx_z) = xz;
        g.at(f.vz_x) = zx;
        g.at(f.vz_z) = zz;
        vx = xx + xz;
        vz = zx + zz;
    } else {
        vx = v.p + (kx * t.a + kz * t.b);
        vz = v.q + (kx * t.e + kz * t.d);
    }
    g.at(f.vx) = vx;
    g.at(f.vz) = vz;
}

// State of a stress update: the six splits of damped cells, the components of
// the others (BARE: without the source, kept in txx_x, tzz_z, txz_x).
template <typename T, bool BARE>
struct StressState {
    T a, b, e, az, bz, ez;
    __device__ __forceinline__ void load(const GradTile& g, const EFieldT<T>& f) {
        a = b = e = az = bz = ez = T(0);
        if (!g.upd()) return;
        a = g.at(BARE ? f.txx_x : f.txx);
        b = g.at(BARE ? f.tzz_z : f.tzz);
        e = g.at(BARE ? f.txz_x : f.txz);
        if (g.damped()) {
            a = g.at(f.txx_x);
            b = g.at(f.tzz_x);
            e = g.at(f.txz_x);
            az = g.at(f.txx_z);
            bz = g.at(f.tzz_z);
            ez = g.at(f.txz_z);
        }
    }
};
// Moduli and image of a cell in the wavefield's precision.
template <typename T>
struct Cell {
    T l, mu, l2m, mp, ms;
    __device__ __forceinline__ Cell(float lam, float mu_, float dmp, float dms)
        : l(lam), mu(mu_), l2m((T)lam + 2 * (T)mu_), mp(-(T)dmp), ms(-(T)dms) {}
};
// Born source of the velocities behind e (born.cu:351-405): added to (txx, tzz, txz).
template <typename T>
__device__ __forceinline__ void born_source(const Cell<T>& m, T ix, T iz, const Taps<T>& e, T& xx, T& zz, T& xz) {
    const T p = 2 * m.l2m * m.mp, q = 2 * (m.l2m * m.mp - 2 * m.mu * m.ms);
    xx += p * e.xx * ix + q * e.zz * iz;
    zz += q * e.xx * ix + p * e.zz * iz;
    xz += 2 * m.mu * m.ms * (e.xz * ix + e.zx * iz);
}
// Stress step (born.cu:282-349) of an updated cell when step, and the Born
// source of the strains sv on top when src (of cells of the physical window).
template <typename T, bool BARE>
__device__ __forceinline__ void stress_cell(const GradTile& g, const EFieldT<T>& f, const StressState<T, BARE>& s,
                                            const DampState& ds, const Cell<T>& m, T dt, const Ratios<T>& q,
                                            bool step, const Taps<T>& e, bool src, const Taps<T>& sv) {
    const T kx = q.kx, kz = q.kz;
    if (g.damped()) {
        if (!step) return;  // no source outside the physical window
        const Damp<T> d(ds.x, ds.z, dt);
        const T a1 = (d.d1 * s.a + kx * m.l2m * e.xx) * d.r2, a2 = (d.d3 * s.az + kz * m.l * e.zz) * d.r4;
        const T b1 = (d.d1 * s.b + kx * m.l * e.xx) * d.r2, b2 = (d.d3 * s.bz + kz * m.l2m * e.zz) * d.r4;
        const T e1 = (d.d1 * s.e + kx * m.mu * e.xz) * d.r2, e2 = (d.d3 * s.ez + kz * m.mu * e.zx) * d.r4;
        g.at(f.txx_x) = a1;
        g.at(f.txx_z) = a2;
        g.at(f.tzz_x) = b1;
        g.at(f.tzz_z) = b2;
        g.at(f.txz_x) = e1;
        g.at(f.txz_z) = e2;
        g.at(f.txx) = a1 + a2;
        g.at(f.tzz) = b1 + b2;
        g.at(f.txz) = e1 + e2;
        return;
    }
    T xx = s.a, zz = s.b, xz = s.e;
    if (step) {
        xx += kx * m.l2m * e.xx + kz * m.l * e.zz;
        zz += kx * m.l * e.xx + kz * m.l2m * e.zz;
        xz += m.mu * (kx * e.xz + kz * e.zx);
        g.at(BARE ? f.txx_x : f.txx) = xx;
        g.at(BARE ? f.tzz_z : f.tzz) = zz;
        g.at(BARE ? f.txz_x : f.txz) = xz;
    }
    if (BARE) {
        if (src && g.interior()) born_source(m, q.ix, q.iz, sv, xx, zz, xz);
        g.at(f.txx) = xx;
        g.at(f.tzz) = zz;
        g.at(f.txz) = xz;
    }
}

// vz and vx of a receiver cell into every trace that records its column.
template <typename T>
__device__ __forceinline__ void record_cell(const SlotDesc& S, const int* rmap, const int* rnext, int ix, int nt,
                                            int it, T vz, T vx, float* rz, float* rx) {
    for (int r = rmap[S.rmap_off + ix]; r >= 0; r = rnext ? rnext[S.rix_off + r] : -1) {
        const size_t o = (size_t)S.rec_off + (size_t)r * nt + it;
        rz[o] = (float)vz;
        rx[o] = (float)vx;
    }
}

// Velocity of f at step it on a tile, with its records and edge bands (ex, ez, or null).
template <typename T>
__device__ __forceinline__ void velocity_tile(const GradTile& g, T* l, const EFieldT<T>& f, const Med& m,
                                              const GradArgs& a, int it, bool source, T* ex, T* ez, float* rec_z,
                                              float* rec_x) {
    Stress3<T> s;
    VelState<T> v;
    DampState ds;
    MedState rho;
    s.load(g, f.txx, f.tzz, f.txz);
    v.load(g, f);
    rho.load(g, m.rho);
    ds.load(g, m);
    s.put(g, l);
    __syncthreads();
    const T dt = a.dt;
    const Ratios<T> q = ratios<T>(a);
    const bool row = source && g.z == g.S.isz, rec = rec_z && g.z == g.S.igz;
    if (!g.own()) return;
    Grad4<T> t(g, s, l);
    // the source sample, on txx and tzz of the source cell for this update only
    const int far = g.S.isx - g.col();
    if (source && (unsigned)(far + 3) < 8u) {
        const T w = a.wav[it];
        if (row) t.a += w * tap<T>(far);
        if (far == 0) t.d += w * tap<T>(g.S.isz - g.z);
    }
    if (!g.zupd) return;
    const T br = T(1) / (T)rho.v;
    T vx, vz;
    velocity_cell(g, f, v, ds, dt, br * q.kx, br * q.kz, t, vx, vz);
    if (ex) {
        const int e = band_place(g.S, g.col(), g.z);
        if (e >= 0) {
            const long long base = g.S.edge_off + it * band_step(g.S);
            ex[base + e] = vx;
            ez[base + e] = vz;
        }
    }
    if (rec) record_cell(g.S, a.rmap, a.rnext, g.col(), a.nt, it, vz, vx, rec_z, rec_x);
}

// Stress of f when step, with the Born source of the velocities (svx, svz) on
// top when src.
template <typename T, typename TS, bool BARE>
__device__ __forceinline__ void stress_tile(const GradTile& g, T* l, TS* ls, const EFieldT<T>& f, const Med& m,
                                            const GradArgs& a, bool step, bool src, const TS* svx, const TS* svz) {
    Vel2<T> v{};
    Vel2<TS> w{};
    StressState<T, BARE> s;
    DampState ds;
    MedState lam, mu, dmp, dms;
    if (step) v.load(g, f.vx, f.vz);
    if (BARE && src) w.load(g, svx, svz);
    s.load(g, f);
    lam.load(g, m.lam);
    mu.load(g, m.mu);
    if (BARE) {
        dmp.load(g, m.dmp);
        dms.load(g, m.dms);
    }
    ds.load(g, m);
    if (step) v.put(g, l);
    if (BARE && src) w.put(g, ls);
    __syncthreads();
    if (!g.own()) return;
    const Taps<T> e(g, v, l);
    const Taps<T> sv(BARE ? Taps<TS>(g, w, ls) : Taps<TS>(e));  // derivatives in the source field's precision
    if (!g.zupd) return;
    const Cell<T> c(lam.v, mu.v, BARE ? dmp.v : 0.f, BARE ? dms.v : 0.f);
    stress_cell(g, f, s, ds, c, (T)a.dt, ratios<T>(a), step, e, src, sv);
}

}  // namespace

// Forward launch A of pair k: velocity of bg at step k, b at k-1, b2 at k-2,
// with their records and edge bands.
template <typename TB>
__global__ __launch_bounds__(GTHREADS) void k_grad_fwd_v(GradFields<TB> F, Med m, GradArgs a,
                                                     const SlotDesc* __restrict__ slots, GradGrid gg, int k) {
    __shared__ TB l[2 * GradTile::FS];
    GradTile g;
    if (!g.init(slots, gg)) return;
    const int layer = g.layer, it = k - layer;
    if (it < 0 || it >= a.nt) return;
    TB* E = F.edges ? F.edges + (layer == 0 ? 0 : 2 * a.total_edge) : nullptr;
    if (layer == 0)
        velocity_tile<TB>(g, l, F.bg, m, a, it, true, E, E + a.total_edge, nullptr, nullptr);
    else if (layer == 1)
        velocity_tile<TB>(g, l, F.b, m, a, it, false, E, E + a.total_edge, a.rs_z, a.rs_x);
    else
        velocity_tile<float>(g, (float*)l, F.b2, m, a, it, false, nullptr, nullptr, a.rs2_z, a.rs2_x);
}

// Forward launch B of pair k: stress of bg at step k; of b at k-1 with the
// Born source of bg's step k on top; of b2 at k-2 with that of b's step k-1.
template <typename TB>
__global__ __launch_bounds__(GTHREADS) void k_grad_fwd_s(GradFields<TB> F, Med m, GradArgs a,
                                                     const SlotDesc* __restrict__ slots, GradGrid gg, int k) {
    constexpr int FS = GradTile::FS;
    __shared__ TB l[4 * FS];
    GradTile g;
    if (!g.init(slots, gg)) return;
    const int layer = g.layer, it = k - layer;
    const bool step = it >= 0 && it < a.nt, src = layer > 0 && it + 1 >= 0 && it + 1 < a.nt;
    if (!step && !src) return;
    if (layer == 0)
        stress_tile<TB, TB, false>(g, l, l, F.bg, m, a, true, false, nullptr, nullptr);
    else if (layer == 1)
        stress_tile<TB, TB, true>(g, l, l + 2 * FS, F.b, m, a, step, src, F.bg.vx, F.bg.vz);
    else
        stress_tile<float, TB, true>(g, (float*)(l + 2 * FS), l, F.b2, m, a, step, src, F.b.vx, F.b.vz);
}

// Receiver-side stress (FD2DGPU.cu:725-761, 860-895) of an updated cell; txz_z of
// an undamped one holds what the last sum of txz rounded off.
struct AdjStress {
    float a, b, e, ez;
    __device__ __forceinline__ void load(const GradTile& g, const EField& f) {
        a = b = e = ez = 0.f;
        if (!g.upd()) return;
        a = g.at(f.txx);
        b = g.at(f.tzz);
        e = g.at(f.txz);
        ez = g.at(f.txz_z);
        if (g.damped()) e = g.at(f.txz_x);
    }
    __device__ __forceinline__ void step(const GradTile& g, const EField& f, const DampState& ds, float dt,
                                         float kx, float kz, const Taps<float>& t, float& xx, float& zz,
                                         float& xz) const {
        if (g.damped()) {
            const Damp<float> d(ds.x, ds.z, dt);
            xx = (d.d1 * a - kx * t.xx) * d.r2;
            zz = (d.d3 * b - kz * t.zz) * d.r4;
            const float p = (d.d1 * e - kx * t.xz) * d.r2, q = (d.d3 * ez - kz * t.zx) * d.r4;
            g.at(f.txz_x) = p;
            g.at(f.txz_z) = q;
            xz = p + q;
        } else {
            xx = a - kx * t.xx;
            zz = b - kz * t.zz;
            const float d = -(kx * t.xz + kz * t.zx) - ez;
            xz = e + d;
            g.at(f.txz_z) = (xz - e) - d;
        }
        g.at(f.txx) = xx;
        g.at(f.tzz) = zz;
        g.at(f.txz) = xz;
    }
};

// Backward launch 1 of step k: (0) bg stress one step back on the physical
// window (FD2DGPU.cu:993-1082) with its strains, from the velocities that hold
// step k's edge bands; (1) b velocity of step k+1 one step back
// (FD2DGPU.cu:903-989), then step k's edge bands; (2) receiver-side stress and
// the products the velocities differentiate.
template <typename TB>
__global__ __launch_bounds__(GTHREADS) void k_grad_bwd_1(GradFields<TB> F, Med m, GradArgs a,
                                                     const SlotDesc* __restrict__ slots, GradGrid gg, int k) {
    __shared__ TB l[2 * GradTile::FS];
    GradTile g;
    if (!g.init(slots, gg)) return;
    const int layer = g.layer;
    const long long n = a.n;
    const Ratios<TB> q = ratios<TB>(a);
    const TB kx = q.kx, kz = q.kz;
    if (layer == 0) {
        Vel2<TB> v;
        TB xx, zz, xz;
        MedState lam, mu;
        v.load(g, F.lvx, F.lvz);
        g.load(F.bg.txx, xx);
        g.load(F.bg.tzz, zz);
        g.load(F.bg.txz, xz);
        lam.load(g, m.lam);
        mu.load(g, m.mu);
        v.put(g, l);
        __syncthreads();
        if (!g.own()) return;
        const Taps<TB> e(g, v, l);
        if (!g.zupd || !g.interior()) return;
        const Cell<TB> mt(lam.v, mu.v, 0.f, 0.f);
        g.at(F.bg.txx) = xx - (kx * mt.l2m * e.xx + kz * mt.l * e.zz);
        g.at(F.bg.tzz) = zz - (kx * mt.l * e.xx + kz * mt.l2m * e.zz);
        g.at(F.bg.txz) = xz - mt.mu * (kx * e.xz + kz * e.zx);
        g.at(a.g) = (float)(e.xx * q.ix);
        g.at(a.g + n) = (float)(e.zz * q.iz);
        g.at(a.g + 2 * n) = (float)(e.zx * q.iz) + (float)(e.xz * q.ix);
    } else if (layer == 1) {
        if (k + 1 >= a.nt) return;  // the velocities are step k's already
        Stress3<TB> s;
        TB vx = 0, vz = 0, hx = 0, hz = 0;
        MedState rho;
        s.load(g, F.b.txx, F.b.tzz, F.b.txz);
        rho.load(g, m.rho);
        const int band = F.edges && g.upd() ? band_place(g.S, g.col(), g.z) : -1;
        // the bands replace the field, not the splits that the next step starts from: cells of
        // the physical window inside a band keep the bare velocity in vx_x and vz_z
        const bool held = band >= 0 && k + 2 < a.nt;
        if (g.upd()) {
            vx = g.at(F.b.vx);
            vz = g.at(F.b.vz);
        }
        if (held) {
            hx = g.at(F.b.vx_x);
            hz = g.at(F.b.vz_z);
        }
        s.put(g, l);
        __syncthreads();
        const long long base = g.S.edge_off + k * band_step(g.S) + 2 * a.total_edge;
        if (!g.own()) return;
        const Grad4<TB> t(g, s, l);
        if (!g.zupd) return;
        const bool in = g.interior();
        if (in) {
            const TB br = TB(1) / (TB)rho.v;
            vx = (held ? hx : vx) - (br * kx * t.a + br * kz * t.b);
            vz = (held ? hz : vz) - (br * kx * t.e + br * kz * t.d);
        }
        if (band >= 0) {
            if (in) {
                g.at(F.b.vx_x) = vx;
                g.at(F.b.vz_z) = vz;
            }
            vx = F.edges[base + band];
            vz = F.edges[a.total_edge + base + band];
        }
        if (in || band >= 0) {
            g.at(F.b.vx) = vx;
            g.at(F.b.vz) = vz;
        }
    } else {
        float* lf = (float*)l;
        Vel2<float> v;
        AdjStress s;
        DampState ds;
        MedState lam, mu, dmp, dms, cs;
        v.load(g, F.bk.vx, F.bk.vz);
        s.load(g, F.bk);
        lam.load(g, m.lam);
        mu.load(g, m.mu);
        dmp.load(g, m.dmp);
        dms.load(g, m.dms);
        cs.load(g, a.cs);
        ds.load(g, m);
        v.put(g, lf);
        __syncthreads();
        if (!g.own()) return;
        const Taps<float> e(g, v, lf);
        if (!g.zupd) return;
        float xx, zz, xz;
        s.step(g, F.bk, ds, a.dt, a.kx, a.kz, e, xx, zz, xz);
        const float l0 = lam.v, mu0 = mu.v, l2m = l0 + 2 * mu0;
        g.at(a.wk) = l2m * xx + l0 * zz;
        g.at(a.wk + n) = l2m * zz + l0 * xx;
        g.at(a.wk + 2 * n) = mu0 * xz;
        const float mp = -dmp.v, ms = -dms.v;
        const float cp = 2 * l2m * mp, cx = 2 * (l2m * mp - 2 * mu0 * ms);
        g.at(a.pk) = cp * xx + cx * zz;
        g.at(a.pk + n) = cp * zz + cx * xx;
        g.at(a.pk + 2 * n) = cs.v * xz;
    }
}

// Receiver-side velocity (FD2DGPU.cu:591-682) from the products of its stress;
// add_x and add_z go on top of the sum, and undamped cells that may have such a
// term (held: all with the Born adjoint, else receivers) keep the bare velocity
// in vx_x and vz_z.
template <bool BORN>
struct AdjVel {
    float x, z;    // the components of undamped cells, or (BORN) vx_x and vz_z of all
    float hx, hz;  // vx_x and vz_z on a tile that has the receiver row
    float xx, zz;  // vx_x and vz_z of damped cells
    float xz, zx;  // vx_z and vz_x; of undamped cells, what the last sums of x and z rounded off
    __device__ __forceinline__ void load(const GradTile& g, const EField& f, bool receivers) {
        x = z = hx = hz = xx = zz = xz = zx = 0.f;
        if (!g.upd()) return;
        x = g.at(BORN ? f.vx_x : f.vx);
        z = g.at(BORN ? f.vz_z : f.vz);
        xz = g.at(f.vx_z);
        zx = g.at(f.vz_x);
        if (!BORN && receivers) {
            hx = g.at(f.vx_x);
            hz = g.at(f.vz_z);
        }
        if (!BORN && g.damped()) {
            xx = g.at(f.vx_x);
            zz = g.at(f.vz_z);
        }
    }
    __device__ __forceinline__ void step(const GradTile& g, const EField& f, const DampState& ds, float dt,
                                         float kx, float kz, const Grad4<float>& t, bool held, float add_x,
                                         float add_z) const {
        const float ax = kx * t.a, az = kz * t.b, bx = kx * t.e, bz = kz * t.d;
        float vx, vz;
        if (g.damped()) {
            const Damp<float> d(ds.x, ds.z, dt);
            const float nxx = (d.d1 * (BORN ? x : xx) - ax) * d.r2, nxz = (d.d3 * xz - az) * d.r4;
            const float nzx = (d.d1 * zx - bx) * d.r2, nzz = (d.d3 * (BORN ? z : zz) - bz) * d.r4;
            g.at(f.vx_x) = nxx;
            g.at(f.vx_z) = nxz;
            g.at(f.vz_x) = nzx;
            g.at(f.vz_z) = nzz;
            vx = nxx + nxz;
            vz = nzx + nzz;
        } else {
            const float x0 = !BORN && held ? hx : x, z0 = !BORN && held ? hz : z;
            const float dx = -(ax + az) - xz, dz = -(bx + bz) - zx;
            vx = x0 + dx;
            vz = z0 + dz;
            g.at(f.vx_z) = (vx - x0) - dx;
            g.at(f.vz_x) = (vz - z0) - dz;
            if (held) {
                g.at(f.vx_x) = vx;
                g.at(f.vz_z) = vz;
            }
        }
        g.at(f.vx) = vx + add_x;
        g.at(f.vz) = vz + add_z;
    }
};

// Layers 1 and 2 of backward launch 2 (see there).
template <bool BORN, typename TB>
__device__ __forceinline__ void adjoint_velocity_tile(const GradTile& g, float* lf, const EField& f, const float* w,
                                                      const GradFields<TB>& F, const Med& m, const GradArgs& a, int k) {
    constexpr int FS = GradTile::FS;
    const long long n = a.n;
    Stress3<float> s;
    AdjVel<BORN> v;
    DampState ds;
    float p0, p1, p2, cs, xz, hp, hc, hx, add_x = 0.f, add_z = 0.f;
    const bool in = g.interior();  // formed here: after the barrier it takes the kernel from 61 to 74 VGPRs
    s.load(g, w, w + n, w + 2 * n);
    MedState rho;
    rho.load(g, m.rho);
    if constexpr (BORN) {
        g.load(a.pk, p0);
        g.load(a.pk + n, p1);
        g.load(a.pk + 2 * n, p2);
        g.load(a.cs, cs);
        g.load(F.bk.txz, xz);
        hp = g.halo(a.pk);
        hc = g.halo(a.cs);
        hx = g.halo(F.bk.txz);
    }
    // whether the tile has the receiver row: uniform, so that what such a cell starts from is chosen by value
    const int row = g.S.igz - (g.z - g.lane);
    const bool receivers = !BORN && g.own() && row >= 0 && row < 64;
    bool held = BORN;
    v.load(g, f, receivers);
    if (receivers) {
        float x = 0.f, z = 0.f;
        bool any = false;
        for (int r = a.rmap[g.S.rmap_off + g.col()]; r >= 0; r = a.rnext ? a.rnext[g.S.rix_off + r] : -1) {
            any = true;
            if (k > 0) {
                const size_t o = (size_t)g.S.rec_off + (size_t)r * a.nt + (k - 1);
                z += a.rs_z[o];
                x += a.rs_x[o];
            }
        }
        held = any && g.z == g.S.igz;
        add_x = held ? x : 0.f;
        add_z = held ? z : 0.f;
    }
    ds.load(g, m);
    s.put(g, lf);
    if constexpr (BORN) {
        g.put(lf + 2 * FS, p0, hp);
        g.put(lf + 3 * FS, cs, hc);
        g.put(lf + 4 * FS, xz, hx);
    }
    __syncthreads();
    if (!g.own()) return;
    const Grad4<float> t(g, s, lf);
    const float br = 1.f / rho.v;
    if constexpr (BORN) {
        const float px = xp(lf + 2 * FS + g.place()), p1z = zp(p1), p2z = zm(p2);
        const float *C = lf + 3 * FS + g.place(), *X = lf + 4 * FS + g.place();
        const float odd = DS2D_C1 * (C[0] * (X[0] - X[-64])) + DS2D_C2 * (C[64] * (X[64] - X[-128])) +
                          DS2D_C3 * (C[128] * (X[128] - X[-192])) + DS2D_C4 * (C[192] * (X[192] - X[-256]));
        if (in) {
            add_x = -br * (px * a.ix + p2z * a.iz);
            add_z = -br * (p1z * a.iz + odd * a.ix);
        }
    }
    if (!g.zupd) return;
    v.step(g, f, ds, a.dt, br * a.kx, br * a.kz, t, held, add_x, add_z);
}

// Backward launch 2 of step k: (0) bg velocity one step back, and in PML
// windows the copy of it that holds step k-1's edge bands; (1) receiver-side
// velocity with the residual of step k-1 on top; (2) the receiver-side Born
// field's velocity with the Born adjoint (born.cu:408-527) on top.  txz's x
// derivative there weights both taps with the modulus of the upper one
// (born.cu:514-515), as in the reference.
template <typename TB>
__global__ __launch_bounds__(GTHREADS) void k_grad_bwd_2(GradFields<TB> F, Med m, GradArgs a,
                                                     const SlotDesc* __restrict__ slots, GradGrid gg, int k) {
    constexpr int FS = GradTile::FS;
    __shared__ float lf[5 * FS];
    GradTile g;
    if (!g.init(slots, gg)) return;
    const int layer = g.layer;
    if (layer == 0) {
        MedState rho;
        TB* l = (TB*)lf;
        Stress3<TB> s;
        TB vx = 0, vz = 0, lx = 0, lz = 0;
        s.load(g, F.bg.txx, F.bg.tzz, F.bg.txz);
        rho.load(g, m.rho);
        if (g.upd()) {
            vx = g.at(F.bg.vx);
            vz = g.at(F.bg.vz);
            lx = g.at(F.lvx);
            lz = g.at(F.lvz);
        }
        s.put(g, l);
        __syncthreads();
        const Ratios<TB> q = ratios<TB>(a);
        const TB kx = q.kx, kz = q.kz;
        const long long base = g.S.edge_off + (k - 1) * band_step(g.S);
        if (!g.own()) return;
        const Grad4<TB> t(g, s, l);
        if (!g.zupd) return;
        // bg itself goes on without the bands (its splits do), lv takes them; outside the physical
        // window bg has step k's bands, which the source strains of this step still see
        const bool in = g.interior();
        const TB br = TB(1) / (TB)rho.v;
        vx = in ? vx - (br * kx * t.a + br * kz * t.b) : lx;
        vz = in ? vz - (br * kx * t.e + br * kz * t.d) : lz;
        if (in || F.edges) {
            g.at(F.bg.vx) = vx;
            g.at(F.bg.vz) = vz;
        }
        if (F.edges) {
            const int e = k > 0 ? band_place(g.S, g.col(), g.z) : -1;
            if (e >= 0) {
                vx = F.edges[base + e];
                vz = F.edges[a.total_edge + base + e];
            }
            g.at(F.lvx) = vx;
            g.at(F.lvz) = vz;
        }
        return;
    }
    if (layer == 1)
        adjoint_velocity_tile<false, TB>(g, lf, F.bk, a.wk, F, m, a, k);
    else
        adjoint_velocity_tile<true, TB>(g, lf, F.bb, a.wb, F, m, a, k);
}

// Backward launch 3 of step k: (0) b stress one step back with its strains and
// bg's Born source on top, the illumination and the images against the
// receiver-side field (FD2DGPU.cu:3235-3263, 3333-3349); (1) the receiver-side
// Born field's stress and products and the images against it.
template <typename TB>
__global__ __launch_bounds__(GTHREADS) void k_grad_bwd_3(GradFields<TB> F, Med m, GradArgs a,
                                                     const SlotDesc* __restrict__ slots, GradGrid gg) {
    constexpr int FS = GradTile::FS;
    __shared__ TB l[4 * FS];
    GradTile g;
    if (!g.init(slots, gg)) return;
    const int layer = g.layer;
    const long long n = a.n, W = a.wstride;
    float gs[3], ak[3], w7[5], kp = 0.f, ks = 0.f;
    MedState lam, mu;
    lam.load(g, m.lam);
    mu.load(g, m.mu);
    float* const w0 = a.w7 + (layer ? 5 * W : 0);
    if (g.upd() && g.interior()) {
        const float vp = g.at(m.vp), vs = g.at(m.vs), rho = g.at(m.rho);
#pragma unroll
        for (int i = 0; i < 3; ++i) gs[i] = g.at(a.g + i * n);
#pragma unroll
        for (int i = 0; i < 5; ++i)
            if (i < 2 || layer == 0) w7[i] = g.window(w0 + i * W);
        if (layer == 0) {
            ak[0] = g.at(F.bk.txx);
            ak[1] = g.at(F.bk.tzz);
            ak[2] = g.at(F.bk.txz);
        }
        kp = -2 * vp * vp * rho;
        ks = -2 * vs * vs * rho;
    }
    if (layer == 0) {
        Vel2<TB> v0, v1;
        TB xx, zz, xz;
        MedState dmp, dms;
        v0.load(g, F.bg.vx, F.bg.vz);
        v1.load(g, F.b.vx, F.b.vz);
        g.load(F.b.txx_x, xx);
        g.load(F.b.tzz_z, zz);
        g.load(F.b.txz_x, xz);
        dmp.load(g, m.dmp);
        dms.load(g, m.dms);
        v0.put(g, l);
        v1.put(g, l + 2 * FS);
        __syncthreads();
        const Ratios<TB> q = ratios<TB>(a);
        const TB kx = q.kx, kz = q.kz, ix = q.ix, iz = q.iz;
        if (!g.own()) return;
        const Taps<TB> e0(g, v0, l), e1(g, v1, l + 2 * FS);
        if (!g.zupd || !g.interior()) return;
        const Cell<TB> mt(lam.v, mu.v, dmp.v, dms.v);
        TB sxx = xx - (kx * mt.l2m * e1.xx + kz * mt.l * e1.zz);
        TB szz = zz - (kx * mt.l * e1.xx + kz * mt.l2m * e1.zz);
        TB sxz = xz - mt.mu * (kx * e1.xz + kz * e1.zx);
        g.at(F.b.txx_x) = sxx;
        g.at(F.b.tzz_z) = szz;
        g.at(F.b.txz_x) = sxz;
        born_source(mt, ix, iz, e0, sxx, szz, sxz);
        g.at(F.b.txx) = sxx;
        g.at(F.b.tzz) = szz;
        g.at(F.b.txz) = sxz;
        const float hxx = (float)(e1.xx * ix), hzz = (float)(e1.zz * iz);
        const float hxz = (float)(e1.zx * iz) + (float)(e1.xz * ix);
        const float gxx = gs[0], gzz = gs[1], gxz = gs[2];
        const float axx = ak[0], azz = ak[1], axz = ak[2];
        // background strain x receiver stress, illumination
        g.window(w0) = w7[0] + kp * ((gxx + gzz) * (axx + azz));
        g.window(w0 + W) = w7[1] + ks * (-2 * (gxx * azz + gzz * axx) + gxz * axz);
        const float ux = (float)v0.vx, uz = (float)v0.vz;
        g.window(w0 + 2 * W) = w7[2] + (ux * ux + uz * uz);
        // scattered strain x receiver stress
        g.window(w0 + 3 * W) = w7[3] + kp * ((hxx + hzz) * (axx + azz));
        g.window(w0 + 4 * W) = w7[4] + ks * (-2 * (hxx * azz + hzz * axx) + hxz * axz);
    } else {
        float* lf = (float*)l;
        Vel2<float> v;
        AdjStress s;
        DampState ds;
        v.load(g, F.bb.vx, F.bb.vz);
        s.load(g, F.bb);
        ds.load(g, m);
        v.put(g, lf);
        __syncthreads();
        if (!g.own()) return;
        const Taps<float> e(g, v, lf);
        if (!g.zupd) return;
        const float l0 = lam.v, mu0 = mu.v, l2m = l0 + 2 * mu0;
        float xx, zz, xz;
        s.step(g, F.bb, ds, a.dt, a.kx, a.kz, e, xx, zz, xz);
        g.at(a.wb) = l2m * xx + l0 * zz;
        g.at(a.wb + n) = l2m * zz + l0 * xx;
        g.at(a.wb + 2 * n) = mu0 * xz;
        if (!g.interior()) return;
        // background strain x receiver-side scattered stress
        const float gxx = gs[0], gzz = gs[1], gxz = gs[2];
        g.window(w0) = w7[0] + kp * ((gxx + gzz) * (xx + zz));
        g.window(w0 + W) = w7[1] + ks * (-2 * (gxx * zz + gzz * xx) + gxz * xz);
    }
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
        for (int r = a.rmap[S.rmap_off + ix]; r >= 0; r = a.rnext ? a.rnext[S.rix_off + r] : -1) {
            const size_t o = (size_t)S.rec_off + (size_t)r * a.nt + (a.nt - 1);
            F.bk.vz[c] += a.rs_z[o];
            F.bk.vx[c] += a.rs_x[o];
        }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static GradGrid grad_grid(const BatchShape& b, int layers) {
    GradGrid t{ceil_div(b.nzp - 2 * NOP, GROWS), ceil_div(b.max_nxp - 2 * NOP, GradTile::COLS), layers, 0, 0};
    t.total = t.zt * t.xt * layers * b.nslots;
    t.per_xcd = ceil_div(t.total, 8);
    return t;
}

template <typename TB>
void launch_grad_forward(hipStream_t st, const BatchShape& b, const GradFields<TB>& F, Med m, const GradArgs& a,
                         bool second) {
    const int layers = second ? 3 : 2, end = a.nt + layers - 1;
    const GradGrid g = grad_grid(b, layers);
    const dim3 grid(g.per_xcd * 8), block(GTHREADS);
    for (int k = 0; k < end; ++k) {
        hipLaunchKernelGGL(k_grad_fwd_v<TB>, grid, block, 0, st, F, m, a, b.slots, g, k);
        // the last field's last stress feeds nothing (with b2 there, b's is step nt-1's at k = nt)
        if (k + 1 < end)
            hipLaunchKernelGGL(k_grad_fwd_s<TB>, grid, block, 0, st, F, m, a, b.slots, g, k);
    }
}

template <typename TB>
void launch_grad_backward(hipStream_t st, const BatchShape& b, const GradFields<TB>& F, Med m, const GradArgs& a) {
    const dim3 cells(BZ, BX), all(ceil_div(b.nzp, BZ), ceil_div(b.max_nxp, BX), b.nslots);
    hipLaunchKernelGGL(k_grad_bwd_0<TB>, all, cells, 0, st, F, m, a, b.slots);
    const GradGrid g3 = grad_grid(b, 3), g2 = grad_grid(b, 2);
    const dim3 grid3(g3.per_xcd * 8), grid2(g2.per_xcd * 8), block(GTHREADS);
    for (int k = a.nt - 1; k >= 0; --k) {
        hipLaunchKernelGGL(k_grad_bwd_1<TB>, grid3, block, 0, st, F, m, a, b.slots, g3, k);
        hipLaunchKernelGGL(k_grad_bwd_2<TB>, grid3, block, 0, st, F, m, a, b.slots, g3, k);
        hipLaunchKernelGGL(k_grad_bwd_3<TB>, grid2, block, 0, st, F, m, a, b.slots, g2);
    }
}

template void launch_grad_forward<float>(hipStream_t, const BatchShape&, const GradFields<float>&, Med, const GradArgs&, bool);
template void launch_grad_forward<double>(hipStream_t, const BatchShape&, const GradFields<double>&, Med, const GradArgs&, bool);
template void launch_grad_backward<float>(hipStream_t, const BatchShape&, const GradFields<float>&, Med, const GradArgs&);
template void launch_grad_backward<double>(hipStream_t, const BatchShape&, const GradFields<double>&, Med, const GradArgs&);

}  // namespace ds2d
