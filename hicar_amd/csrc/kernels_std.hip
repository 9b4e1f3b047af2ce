// The standard advection scheme (&physics adv=1) on the device:
//   k_std_wind    adv_std_compute_wind (src/physics/advect.f90:444-492): the
//                 mass fluxes U_m, V_m, W_m and the divisors jacobian*rho and
//                 dz*jacobian*rho of the flux-form update.
//   k_std_stage   one adv_std_advect3d call without the limiter (advect.f90:
//                 259-320): flux3 of the stage state with the winds times
//                 t_factor, applied to the base state.  Mode 1 also writes
//                 the first upwind half step of upwind_flux3 (dumb_q,
//                 adv_fluxcorr.f90:172-175), which depends on the base state
//                 only, so RK3 gets it from its first stage's loads; mode 2
//                 writes only that.
//   k_std_limit   WRF_flux_corr (adv_fluxcorr.f90:37-150) and the last update:
//                 scale_in and scale_out of the tile and one ring of cells,
//                 the normalised, re-merged fluxes and the new state, in one
//                 march.
//   k_std_ring    the cells outside the tile, which every call leaves at the
//                 base state (qfluxes = qold, :298).
// The stage and limiter kernels march up the columns of LDS-staged tiles, one
// species per block, and compute each face flux once (see below).  Every
// evaluation is the same IEEE FP32 expression in the Fortran's order (this
// unit is compiled with -ffp-contract=off), so the results are the bits of a
// strict build of the reference.  Fortran MAX/MIN of two reals are the selects
// a > b ? a : b and a < b ? a : b.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "fdiv.hpp"
#include "std_planes.hpp"

namespace icaradv {

namespace {

typedef uint32_t off;  // an element offset (the host limits a domain to 2^30 cells)

// A block of cells [i_lo, i_hi] x [j_lo, j_hi] (0-based), all levels, cut
// into tiles and chunks of kch levels.
struct Region {
    int i_lo, i_hi, j_lo, j_hi, kch;
    int nbx, nby, nbz;  // tiles along i and j, chunks along k
    int ns;             // species of the launch, one per block
};

// the hardware's max and min (one instruction; a NaN operand is ignored)
__device__ __forceinline__ float hmax(float a, float b)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float hmin(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ float fmx(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ float fmn(float a, float b) { return a < b ? a : b; }

// The quotients of a level.
//
// Every kernel divides by 12 or 60 in flux3 and by jacobian*rho and
// dz*jacobian*rho in the update, and the IEEE sequence is 11 instructions
// (the constants' branches 9).  The forms below give the IEEE quotient from
// a reciprocal wherever their operands are in range; `Guard` collects the
// operands of a level's quotients (about one instruction each), and a wave
// that meets one out of range computes the phase again with the forms that
// hold for every operand.  The winds and divisors are species-invariant:
// k_std_wind checks them once per step (wind_in_range, divisor_in_range) and
// a domain with one out of range takes the general forms throughout.
struct Guard {
    bool bad = false;            // a quotient's estimate is denormal, infinite or NaN
    uint32_t key = 0xffffffffu;  // smallest non-zero |numerator| (nz_key)
    // numerators of at least 2^-96 over divisors in [2^-30, 2^30]: exact
    // remainders (2^-101) and normal quotients
    __device__ __forceinline__ bool failed() const
    {
        return bad || key < ((127u - 96u) << 24) - 1u;
    }
};
constexpr int NOT_REGULAR = 0x297;  // class mask: NaN, infinities, denormals
constexpr int NOT_FINITE = 0x207;   // NaN, infinities

// a wind component and its third (the RK3 factors scale it by 0.333 .. 1)
__device__ __forceinline__ bool wind_in_range(float u)
{
    const float a = fabsf(u);
    return a == 0.0f || (a >= 0x1p-100f && a <= 0x1p40f);
}
__device__ __forceinline__ bool divisor_in_range(float r) { return r >= 0x1p-30f && r <= 0x1p30f; }

// x / C for the constants C = 12 and 60 of flux3, with R = 1/C rounded: the
// quotient estimate q = x*R, its remainder negated, q*C - x (exact in one FMA),
// and q - (that)*R rounded once; so a zero x keeps its sign.  Compared with the
// IEEE division over every float for both constants, this returns the IEEE
// quotient for each x with |x| >= 2^-124 and for +-0.  F: the guard
// takes x whose estimate is not a normal number or zero; otherwise smaller x,
// infinities and NaNs take the IEEE division, a branch the lanes of a wave
// skip unless one needs it.
template <int C, bool F>
__device__ __forceinline__ float div_const(float x, Guard &g)
{
    constexpr float R = 1.0f / (float)C;
    if (!F) {
        const uint32_t a = __float_as_uint(x) & 0x7fffffffu;
        if (__builtin_expect(a - 1u < 0x017fffffu || a >= 0x7f800000u, 0)) return x / (float)C;
    }
    const float q = x * R;
    if (F) g.bad |= __builtin_amdgcn_classf(q, NOT_REGULAR);
    return __builtin_fmaf(-__builtin_fmaf(q, (float)C, -x), R, q);
}

// |u| / C for a wind (F: in range, k_std_wind)
template <int C, bool F>
__device__ __forceinline__ float wind_const(float u, Guard &g)
{
    const float x = fabsf(u);
    if (!F) return div_const<C, false>(x, g);
    constexpr float R = 1.0f / (float)C;
    const float q = x * R;
    return __builtin_fmaf(__builtin_fmaf(-q, (float)C, x), R, q);
}

// x / d with y = recip_nr(d) (F) and d in range
template <bool F>
__device__ __forceinline__ float div_by(float x, float d, float y, Guard &g)
{
    if (!F) return x / d;
    g.key = min(g.key, nz_key(x));
    return div_y(x, d, y);
}

// flux3's face formulas (advect.f90:150-178): m3..p2 are q at offsets -3..+2
// from the cell on the positive side of the face.
__device__ __forceinline__ float face_up(float u, float m1, float p0)
{
    return ((u + fabsf(u)) * m1 + (u - fabsf(u)) * p0) / 2.0f;
}

template <bool F>
__device__ __forceinline__ float face_o3(float u, float m2, float m1, float p0, float p1, Guard &g)
{
    float f = 7.0f * (p0 + m1) - (p1 + m2);
    f = div_const<12, F>(u * f, g);
    f = f - wind_const<12, F>(u, g) * (3.0f * (p0 - m1) - (p1 - m2));
    return f;
}

template <bool F>
__device__ __forceinline__ float face_o5(float u, float m3, float m2, float m1, float p0,
                                         float p1, float p2, Guard &g)
{
    float f = 37.0f * (p0 + m1) - 8.0f * (p1 + m2) + (p2 + m3);
    f = div_const<60, F>(u * f, g);
    f = f - wind_const<60, F>(u, g) * (10.0f * (p0 - m1) - 5.0f * (p1 - m2) + (p2 - m3));
    return f;
}

// horizontal face whose positive-side cell is c, stride s (q: a raw pointer
// with signed offsets, or a G<float> with 32-bit ones)
template <int H, bool F, class A, class I, class J>
__device__ __forceinline__ float face_h(float u, const A &q, I c, J stride, Guard &g)
{
    const I s = (I)stride;
    if constexpr (H == 1) {
        return face_up(u, q[c - s], q[c]);
    } else if constexpr (H == 3) {
        return face_o3<F>(u, q[c - 2 * s], q[c - s], q[c], q[c + s], g);
    } else {
        return face_o5<F>(u, q[c - 3 * s], q[c - 2 * s], q[c - s], q[c], q[c + s], q[c + 2 * s], g);
    }
}

// one upwind half step of upwind_flux3 (adv_fluxcorr.f90:160-165)
__device__ __forceinline__ float half_up(float u, float m1, float p0)
{
    return 0.5f * ((u + fabsf(u)) * m1 + (u - fabsf(u)) * p0) / 2.0f;
}

// vertical face kf (1..nz-1) from the window z[m] = q(kf-3+m), m = 0..5
// (advect.f90:180-241): the faces next to the ground and the top stay
// upwind, 5th order falls back to 3rd one face further in.  Window entries
// outside the column are never read by the formula chosen.
template <int V, bool F>
__device__ __forceinline__ float face_vw(float w, const float (&z)[6], int kf, int nz, Guard &g)
{
    if (V == 1 || kf == 1 || kf == nz - 1) return face_up(w, z[2], z[3]);
    if (V == 5 && kf >= 3 && kf <= nz - 3)
        return face_o5<F>(w, z[0], z[1], z[2], z[3], z[4], z[5], g);
    return face_o3<F>(w, z[1], z[2], z[3], z[4], g);
}

// The flux-form update of adv_std_advect3d (advect.f90:301-309); yj, ydj: the
// reciprocals of the divisors (F).
template <bool F>
__device__ __forceinline__ float flux_update(float q0, float xw, float xe, float ys, float yn,
                                             float zb, float zt, float rj, float rdj, float yj,
                                             float ydj, Guard &g)
{
    float r = q0 - div_by<F>((xe - xw) + (yn - ys), rj, yj, g);
    r = r - div_by<F>(zt - zb, rdj, ydj, g);
    if (F) g.bad |= __builtin_amdgcn_classf(r, NOT_FINITE);
    return r;
}

// phase(std::integral_constant<bool, F>, Guard&) with the fast forms where
// `ok`, and again with the general ones if an operand was out of range.  Both
// write the same results wherever both hold.  Returns whether the fast forms
// stand.
template <class P>
__device__ __forceinline__ bool guarded(bool ok, P &&phase)
{
    bool general = true;
    if (ok) {
        Guard g;
        phase(std::integral_constant<bool, true>{}, g);
        general = __any(g.failed());
    }
    if (general) {
        Guard g;
        phase(std::integral_constant<bool, false>{}, g);
    }
    return !general;
}

// A merged flux m through a face, normalised as adv_fluxcorr.f90:129-145
// does: pos / neg are the (scale_in, scale_out) of the cells on the positive
// and negative side of the face.
__device__ __forceinline__ float limit_face(float m, float2 pos, float2 neg)
{
    if (m > 0.0f) return fmn(pos.x, neg.y) * m;
    if (m < 0.0f) return fmn(pos.y, neg.x) * m;
    return m;
}

// Both half steps of upwind_flux3 through one face (adv_fluxcorr.f90:
// 158-185): the first from q, the second added from dumb_q.
__device__ __forceinline__ float up2(float u, float qm, float qp, float dm, float dp)
{
    float f = half_up(u, qm, qp);
    f = f + half_up(u, dm, dp);
    return f;
}

// one thread per cell: 64 along i by 4 along k per block, a row j per block column
struct Cell {
    int i, k, j;
    off c;
};

__device__ __forceinline__ Cell this_cell(const Dims &d)
{
    Cell p;
    p.i = blockIdx.x * 64 + threadIdx.x;
    p.k = blockIdx.y * 4 + threadIdx.y;
    p.j = blockIdx.z;
    p.c = (off)p.i + (off)d.nx * ((off)p.k + (off)d.nz * p.j);
    return p;
}

// ---------------------------------------------------------------------------
// adv_std_compute_wind
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
    k_std_wind(Dims d, float dx, float dt, int adv_den, DomainFields f, float *__restrict__ Um,
               float *__restrict__ Vm, float *__restrict__ Wm, float *__restrict__ Rj,
               float *__restrict__ Rdj, unsigned *__restrict__ general)
{
    const Cell p = this_cell(d);
    if (p.i >= d.nx || p.k >= d.nz) return;
    const off c = p.c, sj = (off)d.nx * d.nz, sz = d.nx;
    const float r0 = adv_den ? f.density[c] : 1.0f;  // :472-473
    const off fu = (off)p.i + (off)(d.nx + 1) * ((off)p.k + (off)d.nz * p.j);
    float um = 0.0f, vm = 0.0f, wm;
    if (p.i >= 1) {  // :478-479, U_m(ims+1:ime)
        const float rw = adv_den ? f.density[c - 1] : 1.0f;
        um = f.u[fu] * dt * (r0 + rw) * 0.5f * f.jaco_u[fu] / dx;
    }
    Um[fu] = um;
    if (p.i == d.nx - 1) Um[fu + 1] = 0.0f;
    if (p.j >= 1) {  // :480-481, V_m(:,:,jms+1:jme)
        const float rs = adv_den ? f.density[c - sj] : 1.0f;
        vm = f.v[c] * dt * (r0 + rs) * 0.5f * f.jaco_v[c] / dx;
    }
    Vm[c] = vm;
    if (p.j == d.ny - 1) Vm[c + sj] = 0.0f;
    if (p.k < d.nz - 1) {  // :475-476 rho_i, :483
        const float ra = adv_den ? f.density[c + sz] : 1.0f;
        const float ri = (r0 * f.dz[c] + ra * f.dz[c + sz]) / (f.dz[c] + f.dz[c + sz]);
        wm = f.w[c] * dt * f.jaco_w[c] * ri;
    } else {  // :484
        wm = f.w[c] * dt * f.jaco_w[c] * r0;
    }
    Wm[c] = wm;
    const float rj = f.jaco[c] * r0, rdj = f.dz[c] * f.jaco[c] * r0;
    Rj[c] = rj;    // jaco*rho of :304
    Rdj[c] = rdj;  // dz*jaco*rho of :309
    if (!(wind_in_range(um) && wind_in_range(vm) && wind_in_range(wm) && divisor_in_range(rj) &&
          divisor_in_range(rdj)))
        *general = 1u;  // the species kernels take the general quotients
}

// ---------------------------------------------------------------------------
// Column marches over tiles staged in LDS
// ---------------------------------------------------------------------------
// A block of 8 waves covers a tile of TJ = 8 RW rows, one lane per column, and
// marches up a chunk of levels; a wave owns RW = 2 adjacent rows, or one on
// grids too small to fill the GPU (launch_std_orders).  Levels
// are staged in LDS as planes with the stencils' halo: each wave its own
// rows, one halo row and the few columns beside its rows; the planes form a
// ring that also serves the vertical stencils, whose topmost level is still
// in the registers that prefetched it.  Then every face is computed once:
//   x  on the west side of each lane's cell (the east face comes from the
//      next lane by a lane move),
//   y  on the south side of each row (the north face of a wave's last row is
//      the next wave's first, passed through LDS),
//   z  above each level (the face under a level is carried in registers).
// The kernels are bound by VALU issue, so besides the scheme's arithmetic
// they hold little else: rows and levels are scalar, a load is a scalar base
// plus one lane offset, rows and columns outside the domain hold clamped
// copies (their values reach no cell that is written) and no lane is masked
// but for the halo columns and the stores.
// Blocks take one species each, the species fastest in the block order and
// the tiles in groups of GY rows, so that the species of a tile and its
// neighbours run close together on one XCD and share its winds, divisors and
// halos in L2 (groups of 1, 2 and 8 rows measured 1-4% slower over a step).
constexpr int NTHR = 64 * NWAVE;
constexpr int SCOLS = 63;       // columns a stage updates (lane 63 supplies a face)
constexpr int LCOLS = 61;       // columns the limiter updates (lanes 1..61)
constexpr int GY = 4;           // tile rows that run side by side

typedef __attribute__((address_space(1))) const char gcchar;
typedef __attribute__((address_space(1))) char gchar;
typedef __attribute__((address_space(1))) const float gcfloat;
typedef __attribute__((address_space(1))) float gfloat;

// element c (uniform) plus a lane's 32-bit offset in bytes.  With an offset the
// compiler knows nothing of (unknown) the base stays in scalar registers and
// the access takes both; one it can widen ahead of the loop takes a 64-bit
// addition per access and register pairs.
__device__ __forceinline__ void unknown(unsigned &o) { asm("" : "+v"(o)); }
// the same for a scalar: sums of it with every base are not kept over the loop
__device__ __forceinline__ void unknown(size_t &o) { asm("" : "+s"(o)); }
__device__ __forceinline__ float gld(const float *p, size_t c, unsigned lane)
{
    return *(gcfloat *)((gcchar *)(gcfloat *)(p + c) + lane);
}
__device__ __forceinline__ void gst(float *p, size_t c, unsigned lane, float v)
{
    *(gfloat *)((gchar *)(gfloat *)(p + c) + lane) = v;
}

// the value of the next lane (lane 63: 0) and of the previous lane (lane 0: 0)
__device__ __forceinline__ float lane_next(float v)
{
    const int b = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x130, 0xf, 0xf, true));  // wave_shl:1
}
__device__ __forceinline__ float lane_prev(float v)
{
    const int b = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x138, 0xf, 0xf, true));  // wave_shr:1
}

// A block's place: species, tile and chunk; lane L holds column ib + L, row r
// of the tile is j0 + r
struct Place {
    Dims d;
    int s, ib, j0, k0, k1;
    int L, w;
    int x0;             // first column of the tile's addresses
    unsigned lane;      // this lane's clamped column - x0, in bytes
    size_t sk, sj;
    // cell (x0, 0, row r), the row clamped to the domain
    __device__ __forceinline__ size_t row(int r) const
    {
        return (size_t)x0 + sj * (size_t)min(max(j0 + r, 0), d.ny - 1);
    }
    // the same in the x-face array (nx + 1 per row)
    __device__ __forceinline__ size_t urow(int r) const
    {
        return (size_t)x0 + (sk + 1) * (size_t)d.nz * (size_t)min(max(j0 + r, 0), d.ny - 1);
    }
    // clamped column ib + c as an offset from x0 in bytes
    __device__ __forceinline__ unsigned col(int c) const
    {
        return (unsigned)(min(max(ib + c, 0), d.nx - 1) - x0) * 4u;
    }
};

// first: the column of lane 0 relative to the tile's first updated column;
// west: the columns staged west of lane 0
template <int COLS, int ROWS>
__device__ __forceinline__ Place place(const Dims &d, const Region &r, int first, int west)
{
    Place p;
    p.d = d;
    unsigned t = xcd_block();
    p.s = (int)(t % (unsigned)r.ns);
    t /= (unsigned)r.ns;
    const int bz = (int)(t % (unsigned)r.nbz);
    t /= (unsigned)r.nbz;
    const unsigned gsz = (unsigned)r.nbx * GY, grp = t / gsz;
    const unsigned rows = min((unsigned)GY, (unsigned)r.nby - grp * GY);
    t -= grp * gsz;
    const int bx = (int)(t / rows), by = (int)(grp * GY + t % rows);
    p.ib = r.i_lo + bx * COLS + first;
    p.j0 = r.j_lo + by * ROWS;
    p.k0 = bz * r.kch;
    p.k1 = min(d.nz, p.k0 + r.kch);
    p.L = (int)threadIdx.x & 63;
    p.w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    p.x0 = max(0, p.ib - west);
    p.sk = (size_t)d.nx;
    p.sj = (size_t)d.nx * d.nz;
    p.lane = p.col(p.L);
    return p;
}

// the flux3 face under level k0 (k0 > 0) of a lane's column, from memory; o:
// the column's cell at level k0
template <int V>
__device__ __forceinline__ float face_under(float w, const float *q, size_t o, unsigned lane, int k0,
                                            int nz, size_t sk)
{
    float z[6];
#pragma unroll
    for (int m = 0; m < 6; m++) {
        const int k = k0 - 3 + m;
        z[m] = k >= 0 && k < nz ? gld(q, o + sk * (size_t)k - sk * (size_t)k0, lane) : 0.0f;
    }
    Guard g;
    return face_vw<V, false>(w, z, k0, nz, g);
}

// One RK3 stage / Euler step over tiles: flux3 of the stage state with the
// winds times t applied to the base state (MODE 0 on the tile; MODE 1 the
// same plus the dumb_q half step on the tile and one ring, where the stage
// state is the base state; MODE 2 dumb_q alone on that region).
// One barrier per level: iteration k reads plane k (x, y) and its own columns
// of the ring (z), stages level k + LA into the slot of the lowest level only
// its own columns read, and passes the y faces through a buffer per parity.
// Measured on 1024 x 1024 x 30, 10 species, h5/v3: mode 0 1.62 ms (7.1 GB,
// 4.4 TB/s: near the rate of a copy), mode 1 1.94 ms (6.4 GB; waiting for
// memory and barriers half of the time), against 1.93 and 2.29 ms for one-row
// waves over 7-row tiles whose quotients took the IEEE sequence.  Six waves
// per SIMD: 80 registers hold mode 1 with a few values in scratch; five waves
// (no scratch) and eight took 2.3 and 3.4 ms.
template <int H, int V, int MODE, int RW>
__global__ void __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(6)))
    k_std_stage(StdGeom g, float t, StdBatch b, Region r)
{
    using T = StagePlanes<H, V, RW>;
    using P = typename T::P;
    constexpr int HH = T::HH, LA = T::LA, TJ = T::TJ;
    constexpr bool FL = MODE <= 1, DQ = MODE >= 1;
    __shared__ float sq[P::WORDS];
    __shared__ float sy[2][NWAVE + 1][64], sh[2][DQ ? NWAVE + 1 : 1][64];
    Place p = place<SCOLS, TJ>(g.d, r, 0, HH);
    const bool ok = *g.general == 0u;  // winds and divisors in range (k_std_wind)
    const int nz = p.d.nz, w = p.w, L = p.L;
    const size_t sk = p.sk, su = p.sk + 1;
    const float *const qin = MODE == 0 ? b.qin[p.s] : b.qold[p.s];
    const float *const qo = b.qold[p.s];
    float *const out = b.out[p.s], *const odq = b.dq[p.s];
    const int ra = RW * w;                           // own rows ra .. ra + RW - 1
    const bool last = w == NWAVE - 1;                // computes the faces north of row TJ - 1
    const bool hx = w < 2 * HH;                      // stages a halo row
    const int rx = w < HH ? w - HH : TJ + w - HH;
    size_t ca[RW], ua[RW];
#pragma unroll
    for (int e = 0; e < RW; e++) {
        ca[e] = p.row(ra + e);
        ua[e] = p.urow(ra + e);
    }
    size_t cx = p.row(hx ? rx : ra), cl = p.row(last ? TJ : ra);
    // columns beside the own rows: lanes 0..7 for row ra, 8..15 for ra + 1.  A
    // lane's element offset from row ra holds in 32 bits, also in bytes (a
    // domain has at most 2^30 cells).
    const int he = L & 7, hr = (L >> 3) & 1;
    const bool hc = L < 8 * RW && he < P::XH;
    const int hcol = he < HH ? he - HH : 64 + he - HH;
    unsigned hoff = (hr ? (unsigned)(ca[RW - 1] - ca[0]) * 4u : 0u) + p.col(hcol);
    const int own = P::at(ra, L), ext = P::at(rx, L), hdst = P::at(ra + hr, hcol);
    const bool cell = L < SCOLS && p.ib + L <= r.i_hi;
    const bool put_x = MODE == 0 ? cell : cell && p.ib + L >= g.its && p.ib + L <= g.ite;

    float n0[RW], nx_, nh;  // level being prefetched: own rows, halo row, halo columns
    auto fetch = [&](int k) {
        if (k >= nz) return;
        const size_t o = sk * (size_t)k;
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) n0[e] = gld(qin, ca[e] + o, p.lane);
        if (hx) {
            unknown(p.lane);
            nx_ = gld(qin, cx + o, p.lane);
        }
        if (hc) {
            unknown(hoff);
            nh = gld(qin, ca[0] + o, hoff);
        }
    };
    auto stage = [&](int k) {
        if (k >= nz) return;
        float *const q = sq + P::level(k);
#pragma unroll
        for (int e = 0; e < RW; e++) q[own + e * P::QC] = n0[e];
        if (hx) q[ext] = nx_;
        if (hc) q[hdst] = nh;
    };
    // winds of a level: x and y faces and the top face of the own rows
    float fu[RW], fv[RW + 1], fw[RW];
    auto winds = [&](int k) {
        const size_t o = sk * (size_t)k;
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) {
            fu[e] = gld(g.Um, ua[e] + su * (size_t)k, p.lane);
            fv[e] = gld(g.Vm, ca[e] + o, p.lane);
            fw[e] = gld(g.Wm, ca[e] + o, p.lane);
        }
        if (last) {
            unknown(p.lane);
            fv[RW] = gld(g.Vm, cl + o, p.lane);
        }
    };

    float fzb[RW], hzb[RW];  // the faces under the level
#pragma unroll
    for (int e = 0; e < RW; e++) {
        fzb[e] = hzb[e] = 0.0f;
        if (p.k0 > 0) {
            const size_t o = ca[e] + sk * (size_t)p.k0;
            const float wb = gld(g.Wm, o - sk, p.lane);
            if (FL) fzb[e] = face_under<V>(wb * t, qin, o, p.lane, p.k0, nz, sk);
            if (DQ) hzb[e] = half_up(wb, gld(qo, o - sk, p.lane), gld(qo, o, p.lane));
        }
    }
    for (int k = max(0, p.k0 - LA + 1); k < min(nz, p.k0 + LA); k++) {
        fetch(k);
        stage(k);
    }
    fetch(p.k0 + LA);
    winds(p.k0);
    __syncthreads();
#pragma unroll 1
    for (int k = p.k0; k < p.k1; k++) {
#pragma unroll
        for (int e = 0; e < RW; e++) {
            unknown(ca[e]);
            unknown(ua[e]);
        }
        unknown(cx);
        unknown(cl);
        const size_t o = sk * (size_t)k;
        const bool top = k == nz - 1;
        const float *const q = sq + P::level(k) + own;  // plane k, row ra, this lane
        float rj[RW], rdj[RW], o0[RW];
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) {
            rj[e] = gld(g.Rj, ca[e] + o, p.lane);
            rdj[e] = gld(g.Rdj, ca[e] + o, p.lane);
            o0[e] = MODE == 0 ? gld(qo, ca[e] + o, p.lane) : q[e * P::QC];
        }
        float z[RW][6];  // q(k-2 .. k+3) of the own columns
#pragma unroll
        for (int m = 0; m < 6; m++)
            if (m >= 3 - LA && m <= 2 + LA) {
                const int a = P::level(k - 2 + m) + own;
#pragma unroll
                for (int e = 0; e < RW; e++) z[e][m] = m == 2 + LA ? n0[e] : sq[a + e * P::QC];
            } else {
                z[0][m] = z[RW - 1][m] = 0.0f;
            }
        // flux3 with the winds times t (advect.f90:285-287) and the first
        // upwind half step (adv_fluxcorr.f90:158-175) through the west faces,
        // the faces above the level and the south faces
        float fx[RW], fz[RW], fy[RW + 1], hxw[RW], hz[RW], hy[RW + 1];
        if (FL)
            guarded(ok, [&](auto F, Guard &gd) {
#pragma unroll
                for (int e = 0; e < RW; e++) {
                    fx[e] = face_h<H, F.value>(fu[e] * t, q, e * P::QC, 1, gd);
                    fz[e] = top ? z[e][2] * (fw[e] * t)  // :253
                                : face_vw<V, F.value>(fw[e] * t, z[e], k + 1, nz, gd);
                    fy[e] = face_h<H, F.value>(fv[e] * t, q, e * P::QC, P::QC, gd);
                }
                if (last) fy[RW] = face_h<H, F.value>(fv[RW] * t, q, RW * P::QC, P::QC, gd);
            });
        if (DQ) {
#pragma unroll
            for (int e = 0; e < RW; e++) {
                const int c = e * P::QC;
                hxw[e] = half_up(fu[e], q[c - 1], q[c]);
                hz[e] = top ? 0.5f * q[c] * fw[e] : half_up(fw[e], q[c], z[e][3]);
                hy[e] = half_up(fv[e], q[c - P::QC], q[c]);
            }
            if (last) hy[RW] = half_up(fv[RW], q[(RW - 1) * P::QC], q[RW * P::QC]);
        }
        const int par = k & 1;
        if (FL) {
            sy[par][w][L] = fy[0];
            if (last) sy[par][NWAVE][L] = fy[RW];
        }
        if (DQ) {
            sh[par][w][L] = hy[0];
            if (last) sh[par][NWAVE][L] = hy[RW];
        }
        stage(k + LA);
        fetch(k + LA + 1);
        if (k + 1 < p.k1) winds(k + 1);
        __syncthreads();
        if (FL) fy[RW] = sy[par][w + 1][L];
        if (DQ) hy[RW] = sh[par][w + 1][L];
        float qn[RW], dn[RW];
        float fe[RW], he_[RW];
#pragma unroll
        for (int e = 0; e < RW; e++) {
            if (FL) fe[e] = lane_next(fx[e]);
            if (DQ) he_[e] = lane_next(hxw[e]);
        }
        guarded(ok, [&](auto F, Guard &gd) {
            constexpr bool FD = F.value;
#pragma unroll
            for (int e = 0; e < RW; e++) {
                const float yj = FD ? recip_nr(rj[e]) : 0.0f, ydj = FD ? recip_nr(rdj[e]) : 0.0f;
                if (FL)
                    qn[e] = flux_update<FD>(o0[e], fx[e], fe[e], fy[e], fy[e + 1], fzb[e], fz[e], rj[e],
                                            rdj[e], yj, ydj, gd);
                if (DQ)
                    dn[e] = flux_update<FD>(o0[e], hxw[e], he_[e], hy[e], hy[e + 1], hzb[e], hz[e], rj[e],
                                            rdj[e], yj, ydj, gd);
            }
        });
#pragma unroll
        for (int e = 0; e < RW; e++) {
            const int j = p.j0 + ra + e;
            unknown(p.lane);
            if (FL && put_x && j <= g.jte && (MODE == 0 || j >= g.jts)) gst(out, ca[e] + o, p.lane, qn[e]);
            if (DQ && cell && j <= r.j_hi) gst(odq, ca[e] + o, p.lane, dn[e]);
            if (FL) fzb[e] = fz[e];
            if (DQ) hzb[e] = hz[e];
        }
    }
}

// The limiter and the last update in one march (WRF_flux_corr and the final
// flux form, adv_fluxcorr.f90:37-150, advect.f90:301-309).  Iteration k
// computes the upwind and flux3 faces of level k, then the scales of level k,
// with which the faces between k-1 and k are limited and level k-1 is
// written, and then the limited x and y faces of level k.  The scales go to
// neighbouring rows through LDS and to neighbouring columns by lane moves;
// nothing but the new state is written.  The scales cover the tile and one
// ring: wave w holds the RW rows from RW w - 1 of the tile on, lane L column ib + L (x
// faces on lanes 0..63, scales on 0..62 of rows -1..LROWS, cells 1..61 of
// rows 0..LROWS-1; the last row supplies its south face only).  Two barriers
// per level.  Bound by VALU issue and the waits at the barriers, with two
// blocks of eight waves per CU; what a level carries to the next is kept small
// (111 registers at h5/v3: the state after the horizontal update instead of
// its parts, one register for the one halo row a wave stages) because spilling
// it took 4.7 ms and keeping it in three-row slots 9.3.  1024 x 1024 x 30, 10
// species, h5/v3: 4.1 ms, against 6.4 ms for two marches that each computed
// the faces, the first writing the scales for the second (and 8 bytes per
// cell and species of device memory).
template <int H, int V, int RW>
__global__ void __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(4, 4)))
    k_std_limit(StdGeom g, StdBatch b, Region r)
{
    using T = LimitPlanes<H, V, RW>;
    using P = typename T::P;
    using B = typename T::B;
    constexpr int HH = T::HH, LA = T::LA, TJ = T::TJ;
    constexpr int LROWS = T::LROWS;  // rows written
    __shared__ float sq[P::WORDS];
    __shared__ float so[B::WORDS], sd[B::WORDS];
    // y faces south of a wave's first row: upwind, flux3, wind
    __shared__ float yu[NWAVE + 1][64], yh[NWAVE + 1][64], yv[NWAVE + 1][64];
    __shared__ float ssi[TJ + 2][64], sso[TJ + 2][64];  // scale_in, scale_out of row r - 2 at [r]
    Place p = place<LCOLS, LROWS>(g.d, r, -1, HH);
    const bool ok = *g.general == 0u;  // winds and divisors in range (k_std_wind)
    const int nz = p.d.nz, w = p.w, L = p.L;
    const size_t sk = p.sk, su = p.sk + 1;
    const float *const qin = b.qin[p.s], *const qo = b.qold[p.s], *const dq = b.dq[p.s];
    float *const out = b.out[p.s];
    const int ra = RW * w - 1;  // own rows ra .. ra + RW - 1
    // halo rows: of qin by waves 1 .. 2HH-1, of qold and dq (row -2) by the last two
    const bool hq = w >= 1 && w <= 2 * HH - 1;
    const int rq = w <= HH ? -1 - w : TJ - 2 + w - HH;
    const bool ho = w == NWAVE - 2, hd = w == NWAVE - 1;
    size_t ca[RW], ua[RW];
#pragma unroll
    for (int e = 0; e < RW; e++) {
        ca[e] = p.row(ra + e);
        ua[e] = p.urow(ra + e);
    }
    size_t cq = p.row(hq ? rq : ra), cb = p.row(-2);
    // columns beside the rows: lanes 0..7 row ra, 8..15 row ra + 1; the first
    // XH of qin, the last two column -1 of dq and of qold.  A lane's element
    // offset from row ra holds in 32 bits, also in bytes (a domain has at
    // most 2^30 cells).
    const int he = L & 7, hr = (L >> 3) & 1;
    const bool hcq = L < 8 * RW && he < P::XH, hcb = L < 8 * RW && he >= 6;
    const int hcol = he < HH ? he - HH : 64 + he - HH;
    const unsigned hrow = hr ? (unsigned)(ca[RW - 1] - ca[0]) * 4u : 0u;
    unsigned hqoff = hrow + p.col(hcol), hboff = hrow + p.col(-1);
    const int hqdst = P::at(ra + hr, hcol), hbdst = B::at(ra + hr, -1);
    const int ownq = P::at(ra, L), ownb = B::at(ra, L);
    const int extq = P::at(rq, L), extb = B::at(-2, L);
    const bool put_x = L >= 1 && L <= LCOLS && p.ib + L <= g.ite;

    // the next level to stage (qin: k + LA, qold and dq: k + 1); a wave has at
    // most one halo row
    float nq[RW], no[RW], nd[RW], nrow, nhq, nhb;
    auto fetch_q = [&](int k) {
        if (k >= nz) return;
        const size_t o = sk * (size_t)k;
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) nq[e] = gld(qin, ca[e] + o, p.lane);
        if (hq) {
            unknown(p.lane);
            nrow = gld(qin, cq + o, p.lane);
        }
        if (hcq) {
            unknown(hqoff);
            nhq = gld(qin, ca[0] + o, hqoff);
        }
    };
    auto stage_q = [&](int k) {
        if (k >= nz) return;
        float *const q = sq + P::level(k);
#pragma unroll
        for (int e = 0; e < RW; e++) q[ownq + e * P::QC] = nq[e];
        if (hq) q[extq] = nrow;
        if (hcq) q[hqdst] = nhq;
    };
    auto fetch_b = [&](int k) {
        if (k >= nz) return;
        const size_t o = sk * (size_t)k;
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) {
            no[e] = gld(qo, ca[e] + o, p.lane);
            nd[e] = gld(dq, ca[e] + o, p.lane);
        }
        if (ho || hd) {
            unknown(p.lane);
            nrow = gld(ho ? qo : dq, cb + o, p.lane);
        }
        if (hcb) {
            unknown(hboff);
            nhb = he == 7 ? gld(qo, ca[0] + o, hboff) : gld(dq, ca[0] + o, hboff);
        }
    };
    auto stage_b = [&](int k) {
        if (k >= nz) return;
        const int s = B::level(k);
#pragma unroll
        for (int e = 0; e < RW; e++) {
            so[s + ownb + e * B::QC] = no[e];
            sd[s + ownb + e * B::QC] = nd[e];
        }
        if (ho) so[s + extb] = nrow;
        if (hd) sd[s + extb] = nrow;
        if (hcb) (he == 7 ? so : sd)[s + hbdst] = nhb;
    };
    float fu[RW], fv[RW], fw[RW];
    auto winds = [&](int k) {
        const size_t o = sk * (size_t)k;
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) {
            fv[e] = gld(g.Vm, ca[e] + o, p.lane);
            fu[e] = gld(g.Um, ua[e] + su * (size_t)k, p.lane);
            fw[e] = gld(g.Wm, ca[e] + o, p.lane);
        }
    };

    // The march starts one level below the chunk: the face under k0 is
    // limited with the scales of k0-1 as well, and ends one level above it.
    const int kb = max(0, p.k0 - 1), ke = min(nz - 1, p.k1);
    float uzb[RW], mzb[RW], wb[RW];  // the face under the level: upwind, merged, wind
#pragma unroll
    for (int e = 0; e < RW; e++) {
        uzb[e] = mzb[e] = wb[e] = 0.0f;
        if (kb > 0) {
            const size_t o = ca[e] + sk * (size_t)kb;
            wb[e] = gld(g.Wm, o - sk, p.lane);
            uzb[e] = up2(wb[e], gld(qo, o - sk, p.lane), gld(qo, o, p.lane), gld(dq, o - sk, p.lane),
                         gld(dq, o, p.lane));
            mzb[e] = face_under<V>(wb[e], qin, o, p.lane, kb, nz, sk) - uzb[e];
        }
    }
    // of the level below: its state after the horizontal fluxes, scales,
    // vertical divisor and its reciprocal, and the limited flux through its lower face
    float ph[RW], psi[RW], pso[RW], prdj[RW], pydj[RW], Fzb[RW];
#pragma unroll
    for (int e = 0; e < RW; e++) {
        ph[e] = Fzb[e] = 0.0f;
        psi[e] = pso[e] = prdj[e] = pydj[e] = 1.0f;
    }
    for (int k = max(0, kb - LA + 1); k < min(nz, kb + LA); k++) {
        fetch_q(k);
        stage_q(k);
    }
    if (w == 0) {  // the outermost rows' neighbours: any number (nothing they give is used)
        yu[NWAVE][L] = yh[NWAVE][L] = yv[NWAVE][L] = 0.0f;
        ssi[0][L] = sso[0][L] = ssi[TJ + 1][L] = sso[TJ + 1][L] = 1.0f;
    }
    if (kb > 0) {  // qold under the first level
        fetch_b(kb - 1);
        stage_b(kb - 1);
    }
    fetch_b(kb);
    stage_b(kb);
    fetch_q(kb + LA);
    fetch_b(kb + 1);
    winds(kb);
    __syncthreads();
    // writes level k: its state after the horizontal fluxes less the vertical
    // flux difference over rdj
    auto write = [&](int k, const float (&Fzt)[RW]) {
        float v[RW];
        guarded(ok, [&](auto F, Guard &gd) {
            constexpr bool FD = F.value;
#pragma unroll
            for (int e = 0; e < RW; e++) {
                v[e] = ph[e] - div_by<FD>(Fzt[e] - Fzb[e], prdj[e], pydj[e], gd);
                if (FD) gd.bad |= __builtin_amdgcn_classf(v[e], NOT_FINITE);
            }
        });
#pragma unroll
        for (int e = 0; e < RW; e++) {
            const int row = ra + e;
            unknown(p.lane);
            if (put_x && row >= 0 && row < LROWS && p.j0 + row <= g.jte)
                gst(out, ca[e] + sk * (size_t)k, p.lane, v[e]);
        }
    };
    bool below_fine = kb == 0;  // the faces under the ground are 0
#pragma unroll 1
    for (int k = kb; k <= ke; k++) {
#pragma unroll
        for (int e = 0; e < RW; e++) {
            unknown(ca[e]);
            unknown(ua[e]);
        }
        unknown(cq);
        unknown(cb);
        const size_t o = sk * (size_t)k;
        const bool top = k == nz - 1;
        const float *const q = sq + P::level(k) + ownq;
        const float *const po = so + B::level(k) + ownb, *const pd = sd + B::level(k) + ownb;
        float rj[RW], rdj[RW];
        unknown(p.lane);
#pragma unroll
        for (int e = 0; e < RW; e++) {
            rj[e] = gld(g.Rj, ca[e] + o, p.lane);
            rdj[e] = gld(g.Rdj, ca[e] + o, p.lane);
        }
        // the upwind fluxes of both half steps and flux3 with t_factor 1; a
        // face is kept as its upwind and its merged flux (:80-85)
        float mx[RW], my[RW], mz[RW], ux[RW], uy[RW], uz[RW];
        bool sfin;
        {
            float hx[RW], hy[RW], hz[RW];
            const bool fine = guarded(ok, [&](auto F, Guard &gd) {
#pragma unroll
                for (int e = 0; e < RW; e++) {
                    const int c = e * P::QC;
                    hy[e] = face_h<H, F.value>(fv[e], q, c, P::QC, gd);
                    hx[e] = face_h<H, F.value>(fu[e], q, c, 1, gd);
                    if (top) {
                        hz[e] = q[c] * fw[e];
                    } else {
                        float z[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int m = 3 - LA; m <= 2 + LA; m++)
                            z[m] = m == 2 + LA ? nq[e] : sq[P::level(k - 2 + m) + ownq + c];
                        hz[e] = face_vw<V, F.value>(fw[e], z, k + 1, nz, gd);
                    }
                }
            });
#pragma unroll
            for (int e = 0; e < RW; e++) {
                const int c = e * B::QC;
                const float o0 = po[c], d0 = pd[c];
                uy[e] = up2(fv[e], po[c - B::QC], o0, pd[c - B::QC], d0);
                ux[e] = up2(fu[e], po[c - 1], o0, pd[c - 1], d0);
                if (top) {  // :169, :184
                    uz[e] = 0.5f * o0 * fw[e];
                    uz[e] = uz[e] + 0.5f * d0 * fw[e];
                } else {
                    uz[e] = up2(fw[e], o0, no[e], d0, nd[e]);
                }
                mx[e] = hx[e] - ux[e];
                my[e] = hy[e] - uy[e];
                mz[e] = hz[e] - uz[e];
            }
            // The wave's merged faces of this level and of the one below are
            // numbers.  Where a face has a quotient its guard says so; an
            // upwind face (face_up: first order, next to the ground and the
            // top) has none, and the stage state can hold NaN where the base
            // state is finite.  The sum is not a number if one of them is not
            // (one that overflows costs the general forms, no more).  Checked
            // at every level this took 0.9% of a step at h5/v3.
            bool numbers = fine;
            if (H == 1 || V == 1 || k == 0 || k >= nz - 2) {
                bool nan = false;
#pragma unroll
                for (int e = 0; e < RW; e++)
                    nan |= __builtin_amdgcn_classf((mx[e] + my[e]) + mz[e], NOT_FINITE);
                numbers = fine && !__any(nan);
            }
            sfin = numbers && below_fine;
            below_fine = numbers;
        }
        yu[w][L] = uy[0];
        yh[w][L] = my[0];
        yv[w][L] = fv[0];
        __syncthreads();

        // the north faces: the own next row's, or the next wave's first
        float si[RW], sc[RW], un[RW], mn[RW], vn[RW];
        float yj[RW], ydj[RW];  // reciprocals of the divisors (used where they are in range)
#pragma unroll
        for (int e = 0; e < RW; e++) {
            yj[e] = recip_nr(rj[e]);
            ydj[e] = recip_nr(rdj[e]);
        }
#pragma unroll
        for (int e = 0; e < RW; e++) {
            un[e] = e + 1 < RW ? uy[RW - 1] : yu[w + 1][L];
            mn[e] = e + 1 < RW ? my[RW - 1] : yh[w + 1][L];
            vn[e] = e + 1 < RW ? fv[RW - 1] : yv[w + 1][L];
        }
#pragma unroll
        for (int e = 0; e < RW; e++) {
            const int c = e * B::QC;
            const float uxe = lane_next(ux[e]), me = lane_next(mx[e]), ue = lane_next(fu[e]);
            const float o0 = po[c], qw = po[c - 1], qs = po[c - B::QC], qn = po[c + B::QC];
            const float qe = lane_next(o0);
            const float mb = mzb[e], uzl = uzb[e];
            // :99-121 the bounds' candidates: the neighbours the winds
            // (unscaled) bring in, else the cell itself; wb is 0 under the
            // first level
            const float vx = fu[e] > 0.0f ? qw : ue < 0.0f ? qe : o0;
            const float vy = fv[e] > 0.0f ? qs : vn[e] < 0.0f ? qn : o0;
            const float vb = wb[e] > 0.0f ? so[B::level(k - 1) + ownb + c] : o0;
            const float vt = !top && fw[e] < 0.0f ? no[e] : o0;
            guarded(sfin, [&](auto F, Guard &gd) {
                constexpr bool FD = F.value;
                // FD: every value here is a number (the faces' check above, the
                // north face's and temp's below), so that the hardware's max and min are the
                // Fortran's but for the sign of a zero, which no result keeps
                auto mx2 = [](float a, float b) { return FD ? hmax(a, b) : fmx(a, b); };
                auto mn2 = [](float a, float b) { return FD ? hmin(a, b) : fmn(a, b); };
                const float qmax = mx2(vt, mx2(vb, mx2(vy, mx2(vx, o0))));
                const float qmin = mn2(vt, mn2(vb, mn2(vy, mn2(vx, o0))));
                const float zero = 0.0f;
                if (FD) gd.bad |= __builtin_amdgcn_classf(mn[e], NOT_FINITE);
                // :75-78 the upwind-only value
                const float temp = flux_update<FD>(o0, ux[e], uxe, uy[e], un[e], uzl, uz[e], rj[e],
                                                   rdj[e], yj[e], ydj[e], gd);
                // :88-96
                float fin = div_by<FD>(-((mn2(zero, me) - mx2(zero, mx[e])) + (mn2(zero, mn[e]) - mx2(zero, my[e]))),
                                       rj[e], yj[e], gd);
                fin = fin - div_by<FD>(mn2(zero, mz[e]) - mx2(zero, mb), rdj[e], ydj[e], gd);
                float fout = div_by<FD>((mx2(zero, me) - mn2(zero, mx[e])) + (mx2(zero, mn[e]) - mn2(zero, my[e])),
                                        rj[e], yj[e], gd);
                fout = fout + div_by<FD>(mx2(zero, mz[e]) - mn2(zero, mb), rdj[e], ydj[e], gd);
                // :124-125
                const float up = qmax - temp, dn = temp - qmin;
                const float di = fin + 1.E-15f, dd = fout + 1.E-15f;
                float a, c2;
                if (FD) {
                    gd.key = min(gd.key, min(nz_key(up), nz_key(dn)));
                    gd.bad |= !(di >= 0x1p-60f && di <= 0x1p30f && dd >= 0x1p-60f && dd <= 0x1p30f);
                    a = div_y(up, di, recip_nr(di));
                    c2 = div_y(dn, dd, recip_nr(dd));
                } else {
                    a = up / di;
                    c2 = dn / dd;
                }
                si[e] = fin > up ? mx2(zero, a) : 1.0f;
                sc[e] = fout > dn ? mx2(zero, c2) : 1.0f;
            });
            ssi[RW * w + 1 + e][L] = si[e];
            sso[RW * w + 1 + e][L] = sc[e];
            wb[e] = fw[e];
        }
        // level k-1: its upper faces limited with the scales of both levels
        if (k > kb) {
            float Fzt[RW];
#pragma unroll
            for (int e = 0; e < RW; e++)
                Fzt[e] = limit_face(mzb[e], make_float2(si[e], sc[e]), make_float2(psi[e], pso[e])) + uzb[e];
            if (k - 1 >= p.k0) write(k - 1, Fzt);
#pragma unroll
            for (int e = 0; e < RW; e++) Fzb[e] = Fzt[e];
        }
        stage_q(k + LA);
        stage_b(k + 1);
        fetch_q(k + LA + 1);
        fetch_b(k + 2);
        if (k < ke) winds(k + 1);
        __syncthreads();

        // the limited x and y faces of level k
        float Fs[RW + 1], hs[RW];
        {
            float2 below = make_float2(ssi[RW * w][L], sso[RW * w][L]);  // row ra - 1
#pragma unroll
            for (int e = 0; e <= RW; e++) {
                const float2 c = e < RW ? make_float2(si[e < RW ? e : 0], sc[e < RW ? e : 0])
                                        : make_float2(ssi[RW * w + 1 + RW][L], sso[RW * w + 1 + RW][L]);
                Fs[e] = e == 0 ? limit_face(my[0], c, below) + uy[0]
                               : limit_face(mn[e ? e - 1 : 0], c, below) + un[e ? e - 1 : 0];
                below = c;
            }
        }
#pragma unroll
        for (int e = 0; e < RW; e++) {
            const float2 c = make_float2(si[e], sc[e]);
            const float2 west = make_float2(lane_prev(si[e]), lane_prev(sc[e]));
            const float Fw = limit_face(mx[e], c, west) + ux[e];
            hs[e] = (lane_next(Fw) - Fw) + (Fs[e + 1] - Fs[e]);
        }
        guarded(ok, [&](auto F, Guard &gd) {
            constexpr bool FD = F.value;
#pragma unroll
            for (int e = 0; e < RW; e++) {
                ph[e] = po[e * B::QC] - div_by<FD>(hs[e], rj[e], yj[e], gd);
                if (FD) gd.bad |= __builtin_amdgcn_classf(ph[e], NOT_FINITE);
            }
        });
#pragma unroll
        for (int e = 0; e < RW; e++) {
            psi[e] = si[e];
            pso[e] = sc[e];
            prdj[e] = rdj[e];
            pydj[e] = ydj[e];
            mzb[e] = mz[e];
            uzb[e] = uz[e];
        }
        if (top && k < p.k1) {  // the model-top flux is merged but not limited (:139-143)
            float Fzt[RW];
#pragma unroll
            for (int e = 0; e < RW; e++) Fzt[e] = mz[e] + uz[e];
            write(k, Fzt);
        }
    }
}

// qold into out outside the tile, and into dq outside the tile plus one ring
// The columns outside the tile, numbered: the rows below and above the
// tile (whole rows), then the columns west and east of it on the tile's rows.
__host__ __device__ inline long long ring_columns(const StdGeom &g)
{
    const long long nx = g.d.nx, ny = g.d.ny, tr = g.jte - g.jts + 1;
    return (long long)g.jts * nx + (ny - 1 - g.jte) * nx + tr * (g.its + (nx - 1 - g.ite));
}

// reset: the step's flag of k_std_wind, which runs after this kernel, or null
__global__ void __launch_bounds__(256)
    k_std_ring(StdGeom g, StdBatch b, int with_dq, unsigned *reset)
{
    if (reset && blockIdx.x + blockIdx.y + threadIdx.x == 0) *reset = 0u;
    const Dims d = g.d;
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const int k = blockIdx.y;
    if (t >= ring_columns(g)) return;
    const long long below = (long long)g.jts * d.nx, above = (long long)(d.ny - 1 - g.jte) * d.nx;
    const int side = g.its + (d.nx - 1 - g.ite);
    int i, j;
    if (t < below) {
        j = (int)(t / d.nx);
        i = (int)(t % d.nx);
    } else if (t < below + above) {
        j = g.jte + 1 + (int)((t - below) / d.nx);
        i = (int)((t - below) % d.nx);
    } else {
        const long long u = t - below - above;
        j = g.jts + (int)(u / side);
        const int m = (int)(u % side);
        i = m < g.its ? m : g.ite + 1 + (m - g.its);
    }
    const bool ext = i >= g.its - 1 && i <= g.ite + 1 && j >= g.jts - 1 && j <= g.jte + 1;
    const off c = (off)i + (off)d.nx * ((off)k + (off)d.nz * j);
    for (int s = 0; s < b.n; s++) {
        const float v = b.qold[s][c];
        b.out[s][c] = v;
        if (b.out2[s]) b.out2[s][c] = v;
        if (with_dq && !ext) b.dq[s][c] = v;
    }
}

dim3 cells_grid(const Dims &d) { return dim3((d.nx + 63) / 64, (d.nz + 3) / 4, d.ny); }

// A region in tiles of cols x rows and nch chunks of levels, one species per
// block.
Region tiles(int i_lo, int i_hi, int j_lo, int j_hi, int nz, int nspecies, int cols, int rows,
             int nch)
{
    Region r{};
    r.i_lo = i_lo;
    r.i_hi = i_hi;
    r.j_lo = j_lo;
    r.j_hi = j_hi;
    r.nbx = (i_hi - i_lo + 1 + cols - 1) / cols;
    r.nby = (j_hi - j_lo + 1 + rows - 1) / rows;
    r.ns = nspecies;
    r.kch = (nz + nch - 1) / nch;
    r.nbz = (nz + r.kch - 1) / r.kch;
    return r;
}

// Rows per wave and chunks of levels of a launch.  Whole columns of two-row
// waves do the least work; a grid with few tiles needs more blocks (chunks,
// which repeat a few levels, and one-row waves, which repeat more halo rows)
// to fill the GPU.  The choice is the cheapest by a model of a CU's time in
// microseconds: the blocks it is given times their levels times what a level
// costs once the CU is full (work), or the rounds of blocks times what a
// level takes a block by itself (alone), whichever is more.  The constants
// are measured: work on 1024 x 1024 x 30 with 10 species, alone on 60 x 50 x
// 30 with 2, where the choice makes the limiter 21 us (one-row waves) instead
// of 32 and a stage 12 instead of 16.
struct LevelCost {
    double work, alone;
    int resident;  // blocks per CU
};

template <class F>
Region choose(int nz, double extra_levels, const LevelCost (&cost)[2], F &&region, int *rows)
{
    constexpr int CUS = 256;
    Region best{};
    double best_t = 1e300;
    for (int rw = 2; rw >= 1; rw--) {
        const LevelCost &c = cost[rw - 1];
        for (int nch = 1; nch == 1 || (nz + nch - 1) / nch >= 3; nch++) {
            const Region r = region(rw, nch);
            const double blocks = (double)r.nbx * r.nby * r.nbz * r.ns, lev = r.kch + extra_levels;
            const double per_cu = std::ceil(blocks / CUS);
            const double t = std::max(per_cu * lev * c.work, std::ceil(per_cu / c.resident) * lev * c.alone);
            if (t < 0.98 * best_t) {
                best_t = t;
                best = r;
                *rows = rw;
            }
            if (blocks > 64.0 * CUS) break;  // the GPU is full many times over
        }
    }
    return best;
}

dim3 tile_grid(const Region &r) { return dim3((unsigned)r.nbx * r.nby * r.nbz * r.ns); }

// what: 0 a stage (mode), 1 the limiter
template <int H, int V, int RW>
void launch_std_rows(hipStream_t s, int what, const Region &r, const StdGeom &g, float t, int mode,
                     const StdBatch &b)
{
    const dim3 tb(NTHR), tg = tile_grid(r);
    if (what == 1) hipLaunchKernelGGL((k_std_limit<H, V, RW>), tg, tb, 0, s, g, b, r);
    else if (mode == 0) hipLaunchKernelGGL((k_std_stage<H, V, 0, RW>), tg, tb, 0, s, g, t, b, r);
    else if (mode == 1) hipLaunchKernelGGL((k_std_stage<H, V, 1, RW>), tg, tb, 0, s, g, t, b, r);
    else hipLaunchKernelGGL((k_std_stage<1, 1, 2, RW>), tg, tb, 0, s, g, t, b, r);
}

template <int H, int V>
void launch_std_orders(hipStream_t s, int what, const StdGeom &g, float t, int mode,
                       const StdBatch &b)
{
    static const LevelCost stage[2] = {{0.8, 2.0, 4}, {1.45, 2.6, 3}};
    static const LevelCost limit[2] = {{1.45, 2.6, 2}, {2.7, 4.0, 2}};
    int rows = 2;
    Region r;
    if (what == 1)  // the tile, with a ring of scales around it
        r = choose(g.d.nz, 3.0, limit, [&](int rw, int nch) {
            return tiles(g.its, g.ite, g.jts, g.jte, g.d.nz, b.n, LCOLS, NWAVE * rw - 3, nch);
        }, &rows);
    else {
        const int ring = mode == 0 ? 0 : 1;  // dumb_q is needed one cell around the tile
        r = choose(g.d.nz, 1.5, stage, [&](int rw, int nch) {
            return tiles(g.its - ring, g.ite + ring, g.jts - ring, g.jte + ring, g.d.nz, b.n, SCOLS,
                         NWAVE * rw, nch);
        }, &rows);
    }
    if (rows == 2) launch_std_rows<H, V, 2>(s, what, r, g, t, mode, b);
    else launch_std_rows<H, V, 1>(s, what, r, g, t, mode, b);
}

template <int H>
void launch_std_v(hipStream_t s, int what, const StdGeom &g, float t, int mode, const StdBatch &b)
{
    if (g.vorder == 1) launch_std_orders<H, 1>(s, what, g, t, mode, b);
    else if (g.vorder == 3) launch_std_orders<H, 3>(s, what, g, t, mode, b);
    else launch_std_orders<H, 5>(s, what, g, t, mode, b);
}

void launch_std(hipStream_t s, int what, const StdGeom &g, float t, int mode, const StdBatch &b)
{
    if (g.horder == 1) launch_std_v<1>(s, what, g, t, mode, b);
    else if (g.horder == 3) launch_std_v<3>(s, what, g, t, mode, b);
    else launch_std_v<5>(s, what, g, t, mode, b);
}

}  // namespace

void launch_std_wind(hipStream_t s, Dims d, float dx, float dt, int adv_den,
                     const DomainFields &f, float *Um, float *Vm, float *Wm, float *Rj,
                     float *Rdj, unsigned *general)
{
    hipLaunchKernelGGL(k_std_wind, cells_grid(d), dim3(64, 4), 0, s, d, dx, dt, adv_den, f, Um, Vm,
                       Wm, Rj, Rdj, general);
}

void launch_std_stage(hipStream_t s, const StdGeom &g, float t_factor, int mode,
                      const StdBatch &b)
{
    launch_std(s, 0, g, t_factor, mode, b);
}

void launch_std_limit(hipStream_t s, const StdGeom &g, const StdBatch &b)
{
    launch_std(s, 1, g, 1.0f, 0, b);
}

void launch_std_ring(hipStream_t s, const StdGeom &g, const StdBatch &b, int with_dq,
                     unsigned *reset)
{
    const long long cols = ring_columns(g);
    if (cols <= 0) return;
    hipLaunchKernelGGL(k_std_ring, dim3((unsigned)((cols + 255) / 256), g.d.nz), dim3(256), 0, s, g,
                       b, with_dq, reset);
}

}  // namespace icaradv
