// The steps ICAR runs next to advect, on the device copies of the fields the
// advection handle already holds:
//   k_balance_w   balance_uvw (src/physics/wind.f90:88-164, update=.false.):
//                 the horizontal mass-flux divergence (calc_divergence with
//                 horz_only, :201-234) and w integrated up each column so
//                 that it balances (calc_w, :166-199).  One thread per
//                 column, threads along i (coalesced rows), the level below
//                 carried in registers, a few levels' loads in flight.
//   k_dt_partials compute_dt (src/main/time_step.f90:51-168) with
//                 use_density=.false.: per block the maxima of |u|, |v|, |w|
//                 over the whole arrays and of the tile's per-cell Courant
//                 rate; the host takes the maximum over blocks and finishes
//                 in FP32 as the reference does (a maximum is exact in any
//                 order, so the result is the reference's bits).
//   k_forcing     the boundary-forced branch of apply_forcing
//                 (src/objects/domain_obj.f90:3493-3503) for one species.
//   k_strip       the halo strips of the species for the halo exchange.
//   k_clamp       enforce_limits (domain_obj.f90:3092-3150) for every species.
// Every expression keeps the Fortran's evaluation order; this unit is
// compiled with -ffp-contract=off.
#include "../../include/icar_adv.h"
#include "common.hpp"

namespace icaradv {

namespace {

// u_met and v_met of a face (wind.f90:222-228) from the wind, its Jacobian and
// the density of the cells on both sides; at the domain's edge (e) from the
// cell next to it (a) and the one behind that (b).
template <bool RHO>
__device__ __forceinline__ float met(float u, float ju, float a, float b, bool e)
{
    if (!RHO) return u * ju;
    return e ? u * ju * (1.5f * a - 0.5f * b) : u * ju * (a + b) / 2.0f;
}

// Only the balance itself runs up the column; what it takes from a level (its
// divergence and divisor) does not depend on the level below, so LB levels'
// loads are issued together.  With a level at a time the column's 3 waves per
// SIMD waited for memory at every level: 517 x 389 x 40 0.212 ms, now 0.115 ms
// (258 MB, 0.055 ms at the rate of a copy).
constexpr int LB = 4;

template <bool RHO>
__global__ void __launch_bounds__(256)
    k_balance_w(Dims d, int i_s, int i_e, int j_s, int j_e, float dx, DomainFields f,
                float *__restrict__ w)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y;
    if (i >= d.nx || j >= d.ny) return;
    const size_t sk = (size_t)d.nx, sj = (size_t)d.nx * d.nz;
    const size_t c0 = ix(d, i, 0, j);
    if (i < i_s || i > i_e || j < j_s || j > j_e) {  // w = 0 outside the balanced columns (:179)
        for (int k = 0; k < d.nz; k++) w[c0 + sk * k] = 0.0f;
        return;
    }
    const float *__restrict__ rho = f.density, *__restrict__ dz = f.dz, *__restrict__ jw = f.jaco_w;
    const float *__restrict__ u = f.u, *__restrict__ ju = f.jaco_u;
    const float *__restrict__ v = f.v, *__restrict__ jv = f.jaco_v;
    const bool west = i == 0, east = i == d.nx - 1, south = j == 0, north = j == d.ny - 1;
    float wb = 0.0f, rib = 0.0f, jwb = 0.0f;  // w, rho_i and jacobian_w of the level below
    for (int k0 = 0; k0 < d.nz; k0 += LB) {
        float dd[LB], den[LB], ri[LB], jl[LB];  // divergence * dz, divisor, rho_i, jacobian_w
#pragma unroll
        for (int b = 0; b < LB; b++) {
            const int k = min(k0 + b, d.nz - 1);  // past the top: the top again, not used
            const size_t c = c0 + sk * k;
            const size_t fu = (size_t)i + (size_t)(d.nx + 1) * ((size_t)k + (size_t)d.nz * j);
            float rc = 0.0f, rw = 0.0f, re = 0.0f, rs = 0.0f, rn = 0.0f, ru = 0.0f, dzu = 0.0f;
            if (RHO) {
                const size_t cu = k < d.nz - 1 ? c + sk : c;
                rc = rho[c];
                rw = rho[west ? c + 1 : c - 1];
                re = rho[east ? c - 1 : c + 1];
                rs = rho[south ? c + sj : c - sj];
                rn = rho[north ? c - sj : c + sj];
                ru = rho[cu];
                dzu = dz[cu];
            }
            const float dzc = dz[c];
            // the west and south faces' cells in the order of the sum
            const float dU = met<RHO>(u[fu + 1], ju[fu + 1], rc, re, east) -
                             met<RHO>(u[fu], ju[fu], west ? rc : rw, west ? rw : rc, west);
            const float dV = met<RHO>(v[c + sj], jv[c + sj], rc, rn, north) -
                             met<RHO>(v[c], jv[c], south ? rc : rs, south ? rs : rc, south);
            dd[b] = (dU + dV) / dx * dzc;  // :232
            jl[b] = jw[c];
            // rho_i(k) = (rho(k)dz(k) + rho(k+1)dz(k+1)) / (dz(k)+dz(k+1)), :177
            ri[b] = RHO && k < d.nz - 1 ? (rc * dzc + ru * dzu) / (dzc + dzu) : 0.0f;
            den[b] = RHO ? jl[b] * (k < d.nz - 1 ? ri[b] : rc) : jl[b];  // :183-192, :195-198
        }
#pragma unroll
        for (int b = 0; b < LB; b++) {
            const int k = k0 + b;
            if (k >= d.nz) break;
            float wc;
            if (RHO)
                wc = k == 0 ? 0.0f - dd[b] / den[b] : ((wb * rib * jwb) - dd[b]) / den[b];
            else
                wc = ((k == 0 ? 0.0f : wb * jwb) - dd[b]) / den[b];
            w[c0 + sk * k] = wc;
            wb = wc;
            rib = ri[b];
            jwb = jl[b];
        }
    }
}

constexpr int DT_BLOCKS = 1024, DT_THREADS = 256;

__device__ __forceinline__ float block_max(float v, float *sm)
{
    sm[threadIdx.x] = v;
    __syncthreads();
    for (int s = DT_THREADS / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sm[threadIdx.x] = fmaxf(sm[threadIdx.x], sm[threadIdx.x + s]);
        __syncthreads();
    }
    const float r = sm[0];
    __syncthreads();
    return r;
}

// A wave takes the rows (k, j) of the grid in turn, 64 columns at a time: the
// arrays' maxima and the tile's Courant rates from one set of loads, without
// an integer division per cell.  517 x 389 x 40: 0.074 -> 0.034 ms (the three
// winds are 97 MB, 0.021 ms at the rate of a copy).
__global__ void __launch_bounds__(DT_THREADS)
    k_dt_partials(Dims d, int its, int ite, int jts, int jte, float dx, const float *__restrict__ u,
                  const float *__restrict__ v, const float *__restrict__ w,
                  const float *__restrict__ dzl, float *__restrict__ part)
{
    __shared__ float sm[DT_THREADS];
    const int lane = threadIdx.x & 63;
    const long long wave = (long long)blockIdx.x * (DT_THREADS / 64) +
                           __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const long long waves = (long long)gridDim.x * (DT_THREADS / 64), rows = (long long)d.nz * (d.ny + 1);
    float mu = 0.0f, mv = 0.0f, mw = 0.0f, m3 = 0.0f;
    for (long long r = wave; r < rows; r += waves) {  // row ny: the last y faces only
        const int j = (int)(r / d.nz), k = (int)(r % d.nz);
        const size_t c0 = ix(d, 0, k, j), sj = (size_t)d.nx * d.nz;
        const size_t u0 = (size_t)(d.nx + 1) * ((size_t)k + (size_t)d.nz * j);
        const size_t cb0 = k == 0 ? c0 : c0 - (size_t)d.nx;  // zoffset, :104-108
        if (j == d.ny) {
            for (int i = lane; i < d.nx; i += 64) mv = fmaxf(mv, fabsf(v[c0 + i]));
            continue;
        }
        const bool tile = j >= jts && j <= jte;
        const float dzk = dzl[k];
#pragma unroll 4
        for (int i = lane; i < d.nx; i += 64) {
            const float uc = fabsf(u[u0 + i]), ue = fabsf(u[u0 + i + 1]);
            const float vc = fabsf(v[c0 + i]), vn = fabsf(v[c0 + sj + i]);
            const float wc = fabsf(w[c0 + i]), wd = fabsf(w[cb0 + i]);
            mu = fmaxf(mu, fmaxf(uc, ue));
            mv = fmaxf(mv, vc);
            mw = fmaxf(mw, wc);
            const float a = fmaxf(uc, ue) / dx;  // :101-126
            const float b = fmaxf(vc, vn) / dx;
            const float e = fmaxf(wc, wd) / dzk;
            if (tile && i >= its && i <= ite) m3 = fmaxf(m3, fmaxf(fmaxf(a, b), e));
        }
    }
    mu = block_max(mu, sm);
    mv = block_max(mv, sm);
    mw = block_max(mw, sm);
    m3 = block_max(m3, sm);
    if (threadIdx.x == 0) {
        part[4 * blockIdx.x + 0] = mu;
        part[4 * blockIdx.x + 1] = mv;
        part[4 * blockIdx.x + 2] = mw;
        part[4 * blockIdx.x + 3] = m3;
    }
}

}  // namespace

void launch_balance_w(hipStream_t s, Dims d, int i_s, int i_e, int j_s, int j_e, float dx,
                      int adv_den, const DomainFields &f, float *w)
{
    const dim3 g((d.nx + 63) / 64, (d.ny + 3) / 4), t(64, 4);
    if (adv_den)
        hipLaunchKernelGGL(k_balance_w<true>, g, t, 0, s, d, i_s, i_e, j_s, j_e, dx, f, w);
    else
        hipLaunchKernelGGL(k_balance_w<false>, g, t, 0, s, d, i_s, i_e, j_s, j_e, dx, f, w);
}

int dt_partial_blocks() { return DT_BLOCKS; }

void launch_dt_partials(hipStream_t s, Dims d, int its, int ite, int jts, int jte, float dx,
                        const float *u, const float *v, const float *w, const float *dzl,
                        float *part)
{
    hipLaunchKernelGGL(k_dt_partials, dim3(DT_BLOCKS), dim3(DT_THREADS), 0, s, d, its, ite, jts,
                       jte, dx, u, v, w, dzl, part);
}

}  // namespace icaradv

namespace icaradv {

namespace {

// apply_forcing for a boundary-forced 3-D variable (domain_obj.f90:3493-3503):
// the forcing advances by its tendency, then the value takes it where the
// filter is 1 and relaxes towards it where the filter is below 1.  dt is
// double precision in the reference (dt%seconds()), so the tendency and the
// relaxation term are formed in FP64 and rounded to FP32 on assignment, as
// the Fortran does; forcing - value is an FP32 difference.
// A wave takes the rows (k, j) in turn, so no cell needs an integer division:
// 517 x 389 x 40 0.046 -> 0.040 ms.
__global__ void __launch_bounds__(256)
    k_forcing(Dims d, double dt, const float *__restrict__ filt, float *__restrict__ q,
              float *__restrict__ fhi, const float *__restrict__ dqdt)
{
    const int lane = threadIdx.x & 63;
    const long long rows = (long long)d.nz * d.ny;
    for (long long r = (long long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
         r < rows; r += (long long)gridDim.x * 4) {
        const size_t c0 = (size_t)r * d.nx, f0 = (size_t)(r / d.nz) * d.nx;
#pragma unroll 4
        for (int i = lane; i < d.nx; i += 64) {
            const size_t c = c0 + i;
            const float f = (float)((double)fhi[c] + ((double)dqdt[c] * dt));
            fhi[c] = f;
            const float rf = filt[f0 + i];
            if (rf == 1.0f)
                q[c] = f;
            else if (rf < 1.0f)
                q[c] = (float)((double)q[c] + ((double)rf * dt / 3600.0) * (double)(f - q[c]));
        }
    }
}

}  // namespace

void launch_forcing(hipStream_t s, Dims d, double dt, const float *filt, float *q, float *fhi,
                    const float *dqdt)
{
    size_t blocks = ((size_t)d.nz * d.ny + 3) / 4;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_forcing, dim3((unsigned)blocks), dim3(256), 0, s, d, dt, filt, q, fhi,
                       dqdt);
}

}  // namespace icaradv

namespace icaradv {

namespace {

// Copies one rectangular strip [i0, i0+ni) x [j0, j0+nj), all levels, of
// every species between the species arrays and a packed buffer, or from one
// handle's species to another's (both strips the same shape).  Elements are
// moved as raw 4- or 2-byte words, so 16-bit storage travels as it is held.
// Buffer order: species, then j, k, i (i fastest): each species' strip is a
// contiguous sub-box of its (i, k, j) array.
__global__ void __launch_bounds__(256)
    k_strip(HaloStrips hs, int nz, long long per_species_cells, int mode)
{
    const long long total = per_species_cells * hs.n;
    for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < total;
         t += (long long)gridDim.x * 256) {
        const int s = (int)(t / per_species_cells);
        long long r = t - (long long)s * per_species_cells;
        const int ii = (int)(r % hs.ni);
        r /= hs.ni;
        const int k = (int)(r % nz);
        const int jj = (int)(r / nz);
        const size_t a = (size_t)(hs.a_i0 + ii) + (size_t)hs.a_nx * ((size_t)k + (size_t)nz * (hs.a_j0 + jj));
        const size_t b = (size_t)(hs.b_i0 + ii) + (size_t)hs.b_nx * ((size_t)k + (size_t)nz * (hs.b_j0 + jj));
        const int es = hs.esize[s];
        char *boff = (char *)hs.buf + (size_t)hs.buf_off[s];
        if (mode == 0) {  // species a -> buffer
            if (es == 4) ((float *)boff)[t - (long long)s * per_species_cells] = ((const float *)hs.a[s])[a];
            else ((uint16_t *)boff)[t - (long long)s * per_species_cells] = ((const uint16_t *)hs.a[s])[a];
        } else if (mode == 1) {  // buffer -> species b
            if (es == 4) ((float *)hs.b[s])[b] = ((const float *)boff)[t - (long long)s * per_species_cells];
            else ((uint16_t *)hs.b[s])[b] = ((const uint16_t *)boff)[t - (long long)s * per_species_cells];
        } else {  // species a -> species b
            if (es == 4) ((float *)hs.b[s])[b] = ((const float *)hs.a[s])[a];
            else ((uint16_t *)hs.b[s])[b] = ((const uint16_t *)hs.a[s])[a];
        }
    }
}

}  // namespace

void launch_strip(hipStream_t s, const HaloStrips &hs, int nz, int mode)
{
    const long long per = (long long)hs.ni * hs.nj * nz;
    const long long total = per * hs.n;
    if (total <= 0) return;
    long long blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_strip, dim3((unsigned)blocks), dim3(256), 0, s, hs, nz, per, mode);
}

}  // namespace icaradv

namespace icaradv {

namespace {

// enforce_limits (domain_obj.f90:3092-3150, the data_3d branch): where a
// species is below zero it becomes zero.  -0.0 and NaN are not below zero
// and stay.  16-bit storage is judged on its bits: a set sign bit with a
// non-zero magnitude that is not a NaN.  One launch for all species (a block
// row each), 16 bytes per thread and load, written back only where a value
// changed: 6 us for a read-only species of 8 M cells against 15 us for a
// launch per species with 4-byte accesses.
__device__ __forceinline__ uint32_t below32(uint32_t v)
{
    return __uint_as_float(v) < 0.0f ? 0u : v;
}

template <uint32_t EXPM, uint32_t MANM>
__device__ __forceinline__ uint32_t below16(uint32_t v)
{
    const bool nan = (v & EXPM) == EXPM && (v & MANM) != 0;
    return (v & 0x8000u) && (v & 0x7fffu) && !nan ? 0u : v;
}

__device__ __forceinline__ uint32_t below_word(uint32_t v, int storage)
{
    if (storage == ICAR_ADV_STORE_F32) return below32(v);
    if (storage == ICAR_ADV_STORE_BF16 || storage == ICAR_ADV_STORE_BF16_SR)
        return below16<0x7f80u, 0x007fu>(v & 0xffffu) | below16<0x7f80u, 0x007fu>(v >> 16) << 16;
    return below16<0x7c00u, 0x03ffu>(v & 0xffffu) | below16<0x7c00u, 0x03ffu>(v >> 16) << 16;
}

__global__ void __launch_bounds__(256) k_clamp(size_t n, SpeciesList l)
{
    const int s = blockIdx.y, storage = l.storage[s];
    uint32_t *q = static_cast<uint32_t *>(l.q[s]);
    const size_t words = storage == ICAR_ADV_STORE_F32 ? n : n / 2, quads = words / 4;
    const size_t t0 = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
    uint4 *q4 = reinterpret_cast<uint4 *>(q);  // device allocations are 256-byte aligned
    for (size_t p = t0; p < quads; p += step) {
        const uint4 v = q4[p];
        const uint4 r = make_uint4(below_word(v.x, storage), below_word(v.y, storage),
                                   below_word(v.z, storage), below_word(v.w, storage));
        if ((r.x ^ v.x) | (r.y ^ v.y) | (r.z ^ v.z) | (r.w ^ v.w)) q4[p] = r;
    }
    for (size_t p = 4 * quads + t0; p < words; p += step) {
        const uint32_t v = q[p], r = below_word(v, storage);
        if (r != v) q[p] = r;
    }
    if (storage != ICAR_ADV_STORE_F32 && (n & 1) && t0 == 0) {  // the last 16-bit element
        uint16_t *h = static_cast<uint16_t *>(l.q[s]);
        h[n - 1] = (uint16_t)below_word(h[n - 1], storage);
    }
}

}  // namespace

void launch_clamp(hipStream_t s, size_t n, const SpeciesList &l)
{
    if (l.n == 0) return;
    size_t blocks = (n / 4 + 255) / 256;
    blocks = blocks < 1 ? 1 : blocks > 16384 ? 16384 : blocks;
    hipLaunchKernelGGL(k_clamp, dim3((unsigned)blocks, l.n), dim3(256), 0, s, n, l);
}

}  // namespace icaradv
