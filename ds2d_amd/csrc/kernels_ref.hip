// Reference-compatible elastic kernels for gfx950, batched over shot slots.
//
// The step of ds2d_batch_forward mode 0 and of the decomposed RTM.  Each
// kernel keeps the reference kernel's loop bounds and per-cell update
// (cited below) but runs every shot of a batch in one launch: blockIdx.z is
// the slot, the block is 64 lanes along contiguous z x 4 rows along x, and
// the two reference launches that write disjoint outputs (vx/vz, txx_tzz/txz)
// are fused into one.
#include "common.hpp"
#include "kernels.hpp"

namespace ds2d {

namespace {

struct Cell {
    int ix, iz;
    size_t c;
};

__device__ __forceinline__ bool cell_in(const SlotDesc& S, int lo, Cell& k) {
    k.iz = blockIdx.x * BZ + threadIdx.x;
    k.ix = blockIdx.y * BX + threadIdx.y;
    if (k.ix < lo || k.ix >= S.nxp - lo || k.iz < lo || k.iz >= S.nzp - lo) return false;
    k.c = (size_t)S.off + (size_t)k.ix * S.nzp + k.iz;
    return true;
}

// Tap sums of the eight-point staggered derivatives.
//  dpx: sum c_i (f[ix+i] - f[ix-i+1])   (forward half-point in x)
//  dmx: sum c_i (f[ix+i-1] - f[ix-i])   (backward half-point in x)
//  dpz / dmz: same along z.
__device__ __forceinline__ float dpx(const float* f, size_t c, int s) {
    return DS2D_C1 * (f[c + s] - f[c]) + DS2D_C2 * (f[c + 2 * s] - f[c - s]) +
           DS2D_C3 * (f[c + 3 * s] - f[c - 2 * s]) + DS2D_C4 * (f[c + 4 * s] - f[c - 3 * s]);
}
__device__ __forceinline__ float dmx(const float* f, size_t c, int s) {
    return DS2D_C1 * (f[c] - f[c - s]) + DS2D_C2 * (f[c + s] - f[c - 2 * s]) +
           DS2D_C3 * (f[c + 2 * s] - f[c - 3 * s]) + DS2D_C4 * (f[c + 3 * s] - f[c - 4 * s]);
}

}  // namespace

// Velocity split update of born.cu:215-279 (update_vx/update_vz).
__global__ __launch_bounds__(256) void k_ref_v(EField f, Med m, const SlotDesc* __restrict__ slots, float dt,
                                               float dx, float dz) {
    const SlotDesc S = slots[blockIdx.z];
    Cell k;
    if (!cell_in(S, NOP, k)) return;
    const size_t c = k.c;
    const int nzp = S.nzp;
    const float d1 = 1.f - dt * m.dampx[c] / 2, d2 = 1.f + dt * m.dampx[c] / 2;
    const float d3 = 1.f - dt * m.dampz[c] / 2, d4 = 1.f + dt * m.dampz[c] / 2;
    const float a = dpx(f.txx, c, nzp);
    const float b = dmx(f.txz, c, 1);
    const float cz = dpx(f.tzz, c, 1);
    const float e = dmx(f.txz, c, nzp);
    const float br = 1.f / m.rho[c];
    const float nvx_x = (d1 * f.vx_x[c] + br * (dt / dx) * a) / d2;
    const float nvx_z = (d3 * f.vx_z[c] + br * (dt / dz) * b) / d4;
    const float nvz_x = (d1 * f.vz_x[c] + br * (dt / dx) * e) / d2;
    const float nvz_z = (d3 * f.vz_z[c] + br * (dt / dz) * cz) / d4;
    f.vx_x[c] = nvx_x; f.vx_z[c] = nvx_z; f.vx[c] = nvx_x + nvx_z;
    f.vz_x[c] = nvz_x; f.vz_z[c] = nvz_z; f.vz[c] = nvz_x + nvz_z;
}

// born.cu:282-349 update_txx_tzz + update_txz.
__global__ __launch_bounds__(256) void k_ref_s(EField f, Med m, const SlotDesc* __restrict__ slots, float dt,
                                               float dx, float dz) {
    const SlotDesc S = slots[blockIdx.z];
    Cell k;
    if (!cell_in(S, NOP, k)) return;
    const size_t c = k.c;
    const int nzp = S.nzp;
    const float d1 = 1.f - dt * m.dampx[c] / 2, d2 = 1.f + dt * m.dampx[c] / 2;
    const float d3 = 1.f - dt * m.dampz[c] / 2, d4 = 1.f + dt * m.dampz[c] / 2;
    const float dvx = dmx(f.vx, c, nzp);
    const float dvz = dmx(f.vz, c, 1);
    const float dvxz = dpx(f.vx, c, 1);
    const float dvzx = dpx(f.vz, c, nzp);
    const float l = m.lam[c], mu = m.mu[c], l2m = l + 2 * mu;
    const float ntxx_x = (d1 * f.txx_x[c] + l2m * (dt / dx) * dvx) / d2;
    const float ntxx_z = (d3 * f.txx_z[c] + l * (dt / dz) * dvz) / d4;
    const float ntzz_x = (d1 * f.tzz_x[c] + l * (dt / dx) * dvx) / d2;
    const float ntzz_z = (d3 * f.tzz_z[c] + l2m * (dt / dz) * dvz) / d4;
    f.txx_x[c] = ntxx_x; f.txx_z[c] = ntxx_z; f.tzz_x[c] = ntzz_x; f.tzz_z[c] = ntzz_z;
    f.txx[c] = ntxx_x + ntxx_z;
    f.tzz[c] = ntzz_x + ntzz_z;
    const float ntxz_x = (d1 * f.txz_x[c] + (dt / dx) * mu * dvzx) / d2;
    const float ntxz_z = (d3 * f.txz_z[c] + (dt / dz) * mu * dvxz) / d4;
    f.txz_x[c] = ntxz_x; f.txz_z[c] = ntxz_z;
    f.txz[c] = ntxz_x + ntxz_z;
}

// FD2DGPU.cu:2039-2049 GPUapplysource on txx and tzz (one thread per slot).
__global__ void k_inject_src(float* txx, float* tzz, const float* __restrict__ wav,
                             const SlotDesc* __restrict__ slots, int nslots, int it) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nslots) return;
    const SlotDesc S = slots[s];
    const size_t c = (size_t)S.off + (size_t)S.isx * S.nzp + S.isz;
    const float w = wav[it];
    txx[c] += w;
    tzz[c] += w;
}

// FD2DGPU.cu:355-365 GPUseisrecord, generalised to a receiver list.
__global__ void k_record(const float* __restrict__ vz, const float* __restrict__ vx, float* rz, float* rx,
                         const int* __restrict__ rix, const SlotDesc* __restrict__ slots, int nt, int it) {
    const SlotDesc S = slots[blockIdx.y];
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= S.ntr) return;
    const size_t c = (size_t)S.off + (size_t)rix[S.rix_off + r] * S.nzp + S.igz;
    const size_t o = (size_t)S.rec_off + (size_t)r * nt + it;
    rz[o] = vz[c];
    rx[o] = vx[c];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static dim3 cell_grid(const BatchShape& b) { return dim3(ceil_div(b.nzp, BZ), ceil_div(b.max_nxp, BX), b.nslots); }

void launch_ref_v(hipStream_t st, const BatchShape& b, EField f, Med m) {
    hipLaunchKernelGGL(k_ref_v, cell_grid(b), dim3(BZ, BX), 0, st, f, m, b.slots, b.dt, b.dx, b.dz);
}
void launch_ref_s(hipStream_t st, const BatchShape& b, EField f, Med m) {
    hipLaunchKernelGGL(k_ref_s, cell_grid(b), dim3(BZ, BX), 0, st, f, m, b.slots, b.dt, b.dx, b.dz);
}
void launch_inject_src(hipStream_t st, const BatchShape& b, float* txx, float* tzz, const float* wav, int it) {
    hipLaunchKernelGGL(k_inject_src, dim3(ceil_div(b.nslots, 64)), dim3(64), 0, st, txx, tzz, wav, b.slots,
                       b.nslots, it);
}
void launch_record(hipStream_t st, const BatchShape& b, const float* vz, const float* vx, float* rz, float* rx,
                   int it) {
    hipLaunchKernelGGL(k_record, dim3(ceil_div(b.max_ntr, 64), b.nslots), dim3(64), 0, st, vz, vx, rz, rx, b.rix,
                       b.slots, b.nt, it);
}

}  // namespace ds2d
