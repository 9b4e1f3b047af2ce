// MPDATA with fused passes: batched over species and domains (kernel_variant
// 1), or one species at a time (0, at the end of this file).
//
// One advect() step of mpdata_order n (adv_mpdata.f90:352-413) becomes
//   k_coef     species-invariant face coefficients of the pseudo-velocities
//              (|U|(1-|U|/avg G), the cross-term wind products and the face
//              sums of G), once per step
//   k_first    the donor-cell pass (upwind_advection, :43-103) for every
//              species in one launch, the Courant numbers of a cell reused
//              across a block's species
//   k_corr     one launch per corrective pass (iord >= 2) for every species:
//              antidiffusive pseudo-velocities (mpdata_fluxes, :105-252),
//              the 1-D FCT limiter in x, y and z (flux_limiter, :254-350 and
//              adv_mpdata_FCT_core.f90) and the donor-cell flux divergence
//              with the limited velocities, fused in one kernel.
// k_courant_b mpdata_compute_wind for every domain of the batch
// k_corr marches upward through the levels of a 60 x 16 or 60 x 8 column tile
// (halo 2, staged in LDS); x/y neighbours come from LDS planes, the z
// direction (including the column-wise FCT) stays in registers of the thread
// that owns the column.  Species are independent inside advect, so a launch
// covers (tile, species) pairs; blocks are mapped so that the species of one
// tile run on the same XCD and share its L2.
//
// Every expression keeps the reference's evaluation order, with IEEE FP32
// division and no contraction (this unit is compiled with
// -ffp-contract=off), so for FP32 storage the result is bit-identical to the
// exact kernels and to a strict IEEE FP32 build of the reference; the speed
// comes from fusion, batching and the per-step invariants, not from cheaper
// arithmetic.  The MPDATA step on rough fields is sensitive to rounding
// order at the 1e-5..1e-3 level (a reordered build of the reference moves
// theta by ~6e-4 in 5 steps), so no reordering is done.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include <type_traits>

#include "../../include/icar_adv.h"
#include "fast.hpp"
#include "fdiv.hpp"
#include "ring.hpp"

namespace icaradv {

namespace {

// ---------------------------------------------------------------------------
// Pointers read from the descriptor tables in device memory are generic to
// the compiler, which would then emit flat loads (64-bit per-lane addresses,
// both memory counters).  Every buffer here is device memory, so the kernels
// view them in the global address space: global loads with a scalar base
// and a 32-bit lane offset.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(1))) const float gcfloat;
typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) const uint16_t gcu16;
typedef __attribute__((address_space(1))) uint16_t gu16;

__device__ __forceinline__ gcfloat *gp(const float *p) { return (gcfloat *)p; }
__device__ __forceinline__ gfloat *gp(float *p) { return (gfloat *)p; }

// ---------------------------------------------------------------------------
// species storage: FP32 or 16-bit (BF16 / FP16) holding value * 2^-e
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool is_bf16(int kind)
{
    return kind == ICAR_ADV_STORE_BF16 || kind == ICAR_ADV_STORE_BF16_SR;
}

// 16 random bits for the stochastic rounding of cell c of species s at step t:
// a counter-based hash (the murmur3 32-bit finaliser of a mixed key), so the
// rounding is deterministic and reproducible off the device.
__device__ __forceinline__ uint32_t sr_bits(uint32_t c, int s, uint32_t t)
{
    uint32_t x = (c * 0x9E3779B1u) ^ ((uint32_t)(s + 1) * 0x85EBCA77u) ^ (t * 0xC2B2AE3Du);
    x ^= x >> 16;
    x *= 0x85EBCA6Bu;
    x ^= x >> 13;
    x *= 0xC2B2AE35u;
    x ^= x >> 16;
    return x & 0xFFFFu;
}

// BF16 bits of x: stochastic rounding with the 16 random bits rnd (sr), else
// round to nearest even; infinities and NaN are kept (a NaN stays a NaN)
__device__ __forceinline__ uint16_t bf16_of(float x, bool sr, uint32_t rnd)
{
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += sr ? rnd : 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// value -> 16-bit storage of value * inv_scale.  The plain kinds round to
// nearest even; the _SR kinds round up with probability equal to the
// discarded fraction of an ulp (rnd: 16 uniform bits), so that increments
// smaller than half an ulp are not lost on average and the flux form keeps
// conserving mass.
__device__ __forceinline__ uint16_t to16(float v, int kind, float inv_scale, uint32_t rnd)
{
    const float x = v * inv_scale;
    if (is_bf16(kind)) return bf16_of(x, kind == ICAR_ADV_STORE_BF16_SR, rnd);
    if (kind == ICAR_ADV_STORE_F16_SR) {
        const float ax = fabsf(x);
        if (ax >= 6.103515625e-05f) {  // FP16 normal range: 13 mantissa bits are dropped
            const uint32_t u = (__float_as_uint(x) + (rnd & 0x1FFFu)) & ~0x1FFFu;
            return __half_as_ushort(__float2half_rz(__uint_as_float(u)));
        }
        // FP16 subnormals are multiples of 2^-24
        const float a = ax * 16777216.0f;
        const float k = floorf(a);
        const float up = ((float)rnd * 1.52587890625e-05f < a - k) ? 1.0f : 0.0f;
        return __half_as_ushort(__float2half_rn(copysignf((k + up) * 5.9604644775390625e-08f, x)));
    }
    return __half_as_ushort(__float2half_rn(x));
}

__device__ __forceinline__ bool is_sr(int kind)
{
    return kind == ICAR_ADV_STORE_BF16_SR || kind == ICAR_ADV_STORE_F16_SR;
}

// The storage kinds a kernel is compiled for: FP32 only; FP32 and the BF16
// kinds; any kind.  A species' kind is the same for a wave, so the kernels
// branch on it around its loads and stores.
constexpr int QK_F32 = 0, QK_BF16 = 1, QK_ANY = 2;

// Accesses of the marching kernels: a scalar element index and the lane's
// offset in elements.  The species' values come in two steps, the raw bits (a
// 32- or 16-bit load) and the conversion where the value is used, so that no
// conversion right after a load makes the wave wait for it.
typedef __attribute__((address_space(1))) const uint32_t gcu32;
typedef __attribute__((address_space(1))) const char gcchar;
typedef __attribute__((address_space(1))) char gchar;

__device__ __forceinline__ float ld1(const float *b, size_t c, unsigned lane)
{
    return *(gcfloat *)((gcchar *)(gcfloat *)(b + c) + lane * 4u);
}

template <int QK>
__device__ __forceinline__ uint32_t ldq(const void *b, size_t c, unsigned lane, int kind)
{
    if (QK == QK_F32 || kind == ICAR_ADV_STORE_F32)
        return *(gcu32 *)((gcchar *)(gcfloat *)((const float *)b + c) + lane * 4u);
    return *(gcu16 *)((gcchar *)(gcu16 *)((const uint16_t *)b + c) + lane * 2u);
}

// the value of ldq's bits
template <int QK>
__device__ __forceinline__ float cvq(uint32_t b, int kind, float scale)
{
    if (QK == QK_F32 || kind == ICAR_ADV_STORE_F32) return __uint_as_float(b);
    if (QK == QK_BF16 || is_bf16(kind)) return __uint_as_float(b << 16) * scale;
    return __half2float(__ushort_as_half((uint16_t)b)) * scale;
}

// the stored bits of a value at a 16-bit kind of the class
template <int QK>
__device__ __forceinline__ uint16_t q16_of(float v, int kind, float inv_scale, uint32_t rnd)
{
    if (QK == QK_BF16) return bf16_of(v * inv_scale, kind == ICAR_ADV_STORE_BF16_SR, rnd);
    return to16(v, kind, inv_scale, rnd);
}

template <int QK>
__device__ __forceinline__ void stq(void *b, size_t c, unsigned lane, int kind, float inv_scale,
                                    float v, uint32_t rnd)
{
    if (QK == QK_F32 || kind == ICAR_ADV_STORE_F32)
        *(gfloat *)((gchar *)(gfloat *)((float *)b + c) + lane * 4u) = v;
    else
        *(gu16 *)((gchar *)(gu16 *)((uint16_t *)b + c) + lane * 2u) =
            q16_of<QK>(v, kind, inv_scale, rnd);
}

// One pass of one species: where to read q0 (and q1) and where to write.
struct SpecPass {
    const void *q0;   // field before the pass (storage kind0)
    const float *q1;  // field after the previous pass (FP32), or nullptr if equal to q0
    void *out;        // result (storage kindo)
    int kind0, kindo;
    float scale0, inv_scaleo;
};

// Entry s of a species table.  The tables change between launches only, so an
// entry that is the same for every lane of a wave (as it is in the kernels)
// comes by scalar loads: read through a plain pointer it would sit in vector
// registers, and with it every address formed from it.
__device__ __forceinline__ SpecPass species(const SpecPass *tab, int s)
{
    typedef __attribute__((address_space(4))) const uint32_t ccu32;
    constexpr int W = sizeof(SpecPass) / 4;
    ccu32 *const w = (ccu32 *)(uintptr_t)(tab + __builtin_amdgcn_readfirstlane(s));
    uint32_t b[W];
#pragma unroll
    for (int e = 0; e < W; e++) b[e] = w[e];
    SpecPass p;
    __builtin_memcpy(&p, b, sizeof(p));
    return p;
}

// One domain of a batched launch (a single handle, or one member of an
// ensemble of unevenly sized domains).  Cell kernels cover 64x4-thread
// blocks of one level; the corrective kernel covers (tile, species) items.
constexpr int MAXP = 16;  // mpdata_order limit
struct DomDesc {
    Dims d;
    unsigned cb0, bx;     // first global cell block; cell blocks along x
    unsigned f0;          // first global block of the donor-cell kernel
    int ftx, fnk, fkch;   // its tiles along x, level chunks and levels per chunk
    int fng, fsb, fsr;    // its species groups: fsr of fsb + 1 species, then of fsb
    unsigned w0;          // first global corrective work item
    int tiles_x, nspec;
    int nks, kch;         // corrective kernel: column chunks along k and levels per chunk
    float dx, dt;
    int advect_density;
    int compensated;      // flux divergence with compensated sums
    DomainFields f;       // raw inputs
    StepFields sf;        // Courant numbers and products (written by k_courant_b)
    float *coef;          // face coefficients (float4 groups)
    unsigned *step;       // [0] steps taken (drives the stochastic rounding); [1] a coefficient
                          // is out of the bounds of the fast quotients (k_coef)
    float *keep;                 // the donor-cell pass copies its FP32 species here (or nullptr)
    const SpecPass *pass[MAXP];  // species table of pass p at index p-1
};

// domain of global cell block b / work item w: the last entry whose first
// block (item) is <= the key
__device__ __forceinline__ int find_dom_cb(const DomDesc *D, int nd, unsigned b)
{
    int lo = 0, hi = nd - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (D[mid].cb0 <= b) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ int find_dom_f(const DomDesc *D, int nd, unsigned b)
{
    int lo = 0, hi = nd - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (D[mid].f0 <= b) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ int find_dom_w(const DomDesc *D, int nd, unsigned w)
{
    int lo = 0, hi = nd - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (D[mid].w0 <= w) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// (i, k, j) of this thread in a 64x4 cell block
__device__ __forceinline__ void cell_of(const DomDesc &D, unsigned b, int &i, int &k, int &j)
{
    const unsigned l = b - D.cb0;
    const unsigned r = l / D.bx;
    i = (int)(l % D.bx) * 64 + (int)threadIdx.x;
    k = (int)(r % (unsigned)D.d.nz);
    j = (int)(r / (unsigned)D.d.nz) * 4 + (int)threadIdx.y;
}

// ---------------------------------------------------------------------------
// mpdata_compute_wind (adv_mpdata.f90:477-504) and the species-invariant
// products, for every domain of the batch; the same expressions as the
// exact Courant kernel, so the same bits.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_courant_b(const DomDesc *__restrict__ DD, int nd)
{
    const unsigned blk = xcd_block();
    const DomDesc &D = DD[find_dom_cb(DD, nd, blk)];
    int i, k, j;
    cell_of(D, blk, i, k, j);
    const Dims d = D.d;
    if (blk == D.cb0 && threadIdx.x + threadIdx.y == 0) D.step[1] = 0u;
    if (i >= d.nx || j >= d.ny) return;
    gcfloat *__restrict__ den = gp(D.f.density), *__restrict__ fu = gp(D.f.u);
    gcfloat *__restrict__ fv = gp(D.f.v), *__restrict__ fw = gp(D.f.w);
    gcfloat *__restrict__ ju = gp(D.f.jaco_u), *__restrict__ jv = gp(D.f.jaco_v);
    gcfloat *__restrict__ jw = gp(D.f.jaco_w), *__restrict__ jc = gp(D.f.jaco);
    gcfloat *__restrict__ dz = gp(D.f.dz);
    gfloat *__restrict__ oU = gp(D.sf.U), *__restrict__ oV = gp(D.sf.V), *__restrict__ oW = gp(D.sf.W);
    gfloat *__restrict__ oG = gp(D.sf.G), *__restrict__ oGz = gp(D.sf.Gz), *__restrict__ oWd = gp(D.sf.Wd);
    const float dt = D.dt, dx = D.dx;
    const int advect_density = D.advect_density;
    const size_t c = ix(d, i, k, j);
    const size_t sj = (size_t)d.nx * d.nz;
    const float rc = advect_density ? den[c] : 1.0f;  // :489-490
    if (i >= 1) {
        const size_t iu = (size_t)i + (size_t)(d.nx + 1) * ((size_t)k + (size_t)d.nz * j);
        const float rl = advect_density ? den[c - 1] : 1.0f;
        oU[c] = fu[iu] * dt * (rc + rl) * 0.5f * ju[iu] / dx;  // :492-493
    } else {
        oU[c] = 0.0f;
    }
    if (j >= 1) {
        const float rs = advect_density ? den[c - sj] : 1.0f;
        oV[c] = fv[c] * dt * (rc + rs) * 0.5f * jv[c] / dx;  // :494-495
    } else {
        oV[c] = 0.0f;
    }
    float Wc;
    if (k < d.nz - 1) {
        const float ru = advect_density ? den[c + d.nx] : 1.0f;
        Wc = fw[c] * dt * jw[c] * (ru + rc) * 0.5f;  // :496-497
    } else {
        Wc = fw[c] * dt * jw[c] * rc;  // :498
    }
    oW[c] = Wc;
    const float jac = jc[c], dnc = den[c], dzc = dz[c];
    oG[c] = jac * dnc;
    oGz[c] = dzc * jac * dnc;
    oWd[c] = Wc / dzc;
}

// ---------------------------------------------------------------------------
// species-invariant parts of the pseudo-velocities, once per step, each
// evaluated exactly as mpdata_fluxes evaluates it (adv_mpdata.f90:139,151,
// 163,180,192,203,221,233,244):
//   CUx = |U|*(1-|U|/(0.5*(G_r+G_l)))   first factor of the face value
//   CVx = (0.5*U)*edge_v                 prefix of each cross term
//   SGx = G_r+G_l                        its divisor
// for the x face left of a cell (x), the y face south of it (y) and the z
// face on top of it (z).  A cross-term prefix is 0 where the reference skips
// the term (its row/level guards); the corrective kernel tests the same
// guards and never uses those entries.  Stored as three float4 groups per
// cell (x, y, z faces) so that the corrective kernel loads a face's four
// values with one 128-bit load.
// ---------------------------------------------------------------------------
enum { CUX = 0, CXV, CXW, SGX, CUY, CYU, CYW, SGY, CUZ, CZU, CZV, SGZ, NCOEF };

__global__ void __launch_bounds__(256) k_coef(const DomDesc *__restrict__ DD, int nd)
{
    const unsigned blk = xcd_block();
    const DomDesc &D = DD[find_dom_cb(DD, nd, blk)];
    int i, k, j;
    cell_of(D, blk, i, k, j);
    const Dims d = D.d;
    if (i >= d.nx || j >= d.ny) return;
    gcfloat *__restrict__ U = gp(D.sf.U), *__restrict__ V = gp(D.sf.V), *__restrict__ Wd = gp(D.sf.Wd);
    gcfloat *__restrict__ G = gp(D.sf.G);
    gfloat *__restrict__ coef = gp(D.coef);
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const size_t N = (size_t)nx * ny * nz;
    const size_t sk = (size_t)nx, sj = (size_t)nx * nz;
    const size_t c = (size_t)i + sk * ((size_t)k + (size_t)nz * j);
    float v[NCOEF];
#pragma unroll
    for (int e = 0; e < NCOEF; e++) v[e] = 0.0f;
    if (i >= 1) {
        const float Uc = U[c], au = fabsf(Uc);
        v[CUX] = au * (1.0f - au / (0.5f * (G[c] + G[c - 1])));
        v[SGX] = G[c] + G[c - 1];
        if (j >= 1 && j <= ny - 2)
            v[CXV] = 0.5f * Uc * ((1.0f / 4.0f) * (V[c] + V[c + sj] + V[c - 1] + V[c - 1 + sj]));
        if (k >= 1 && k <= nz - 2)
            v[CXW] = 0.5f * Uc * ((1.0f / 4.0f) * (Wd[c] + Wd[c - sk] + Wd[c - 1] + Wd[c - 1 - sk]));
    }
    if (j >= 1) {
        const float Vc = V[c], av = fabsf(Vc);
        v[CUY] = av * (1.0f - av / (0.5f * (G[c] + G[c - sj])));
        v[SGY] = G[c] + G[c - sj];
        if (i >= 1 && i <= nx - 2)
            v[CYU] = 0.5f * Vc * ((1.0f / 4.0f) * (U[c + 1] + U[c + 1 - sj] + U[c] + U[c - sj]));
        if (k >= 1 && k <= nz - 2)
            v[CYW] = 0.5f * Vc * ((1.0f / 4.0f) * (Wd[c] + Wd[c - sk] + Wd[c - sj] + Wd[c - sk - sj]));
    }
    if (k <= nz - 2) {
        const float Wc = Wd[c], aw = fabsf(Wc);
        v[CUZ] = aw * (1.0f - aw / (0.5f * (G[c + sk] + G[c])));
        v[SGZ] = G[c + sk] + G[c];
        if (i >= 1 && i <= nx - 2)
            v[CZU] = 0.5f * Wc * ((1.0f / 4.0f) * (U[c + 1] + U[c + 1 + sk] + U[c] + U[c + sk]));
        if (j >= 1 && j <= ny - 2)
            v[CZV] = 0.5f * Wc * ((1.0f / 4.0f) * (V[c] + V[c + sk] + V[c + sj] + V[c + sk + sj]));
    }
    // outside the bounds the corrective kernel's quotients are proven for
    // (k_corr), it takes the IEEE division for the whole domain
    auto within = [](float c0, float c1, float c2, float sg) {
        return fabsf(c0) <= 16.0f && sg >= 0x1p-30f && sg <= 0x1p30f && fabsf(c1) <= 16.0f * sg &&
               fabsf(c2) <= 16.0f * sg;
    };
    bool ok = true;
    if (i >= 1) ok = ok && within(v[CUX], v[CXV], v[CXW], v[SGX]);
    if (j >= 1) ok = ok && within(v[CUY], v[CYU], v[CYW], v[SGY]);
    if (k <= nz - 2) ok = ok && within(v[CUZ], v[CZU], v[CZV], v[SGZ]) && fabsf(gp(D.f.dz)[c]) <= 0x1p14f;
    if (!ok) D.step[1] = 1u;
#pragma unroll
    for (int g = 0; g < 3; g++)
#pragma unroll
        for (int e = 0; e < 4; e++) coef[4 * ((size_t)g * N + c) + e] = v[4 * g + e];
}

// The time steps of domains d0 .. d0 + n - 1, at both parities of the table.
// They are set in stream order: a step that is still queued reads the ones it
// was enqueued with.
constexpr int DT_SET = 64;
struct DtSet {
    int d0, n;
    float dt[DT_SET];
};
__global__ void __launch_bounds__(DT_SET) k_set_dt(DomDesc *__restrict__ DD, int nd, DtSet v)
{
    const int t = threadIdx.x;
    if (t >= v.n) return;
    DD[v.d0 + t].dt = v.dt[t];
    DD[nd + v.d0 + t].dt = v.dt[t];
}

// one step taken by every domain of the batch (a vector store per domain)
__global__ void __launch_bounds__(64) k_tick(const DomDesc *__restrict__ DD, int nd)
{
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t < nd) DD[t].step[0] = DD[t].step[0] + 1u;
}

// ---------------------------------------------------------------------------
// donor-cell pass for every species (upwind_advection, adv_mpdata.f90:43-103)
// ---------------------------------------------------------------------------
// the value of the next lane (lane 63: 0) and of the previous lane (lane 0:
// 0): one move within the wave, no LDS
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

// x/d: the IEEE division, or (F) the three-operation quotient of fdiv.hpp
template <bool F>
__device__ __forceinline__ float fdiv(float x, float d)
{
    if constexpr (F) return div_y(x, d, recip_nr(d));
    else return x / d;
}

// the same with y = recip_nr(d) computed once for several numerators
template <bool F>
__device__ __forceinline__ float fdiv_y(float x, float d, float y)
{
    if constexpr (F) return div_y(x, d, y);
    else return x / d;
}

// Maxima and minima of values that come from memory.  fmaxf on such a value
// first quiets a possible signalling NaN with an instruction of its own; the
// hardware's max and min ignore quiet NaNs as fmaxf does.
__device__ __forceinline__ float vmax(float a, float b)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmin(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float vmin3(float a, float b, float c)
{
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// max(0, a), min(0, a), and min(1, a, b)
__device__ __forceinline__ float vpos(float a)
{
    float r;
    asm("v_max_f32 %0, 0, %1" : "=v"(r) : "v"(a));
    return r;
}
__device__ __forceinline__ float vneg(float a)
{
    float r;
    asm("v_min_f32 %0, 0, %1" : "=v"(r) : "v"(a));
    return r;
}
__device__ __forceinline__ float vmin1(float a, float b)
{
    float r;
    asm("v_min3_f32 %0, 1.0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// the largest magnitude of a (not negative), b and c
__device__ __forceinline__ float vmax3a(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// flux1 (adv_mpdata.f90:39)
__device__ __forceinline__ float flux1(float l, float r, float U)
{
    return ((U + fabsf(U)) * l + (U - fabsf(U)) * r) / 2.0f;
}

// A block of four waves covers a tile of 62 columns x 8 rows for up to NS
// species and marches up a chunk of levels; a wave holds two adjacent rows, one
// lane per column (lanes 0 and 63 are the neighbours' columns).  So each x face
// is computed once (the east face comes from the next lane), the y face between
// the rows once, the z face above a level is the next level's face below, and a
// level's own values are loaded once: two loads per cell and species and about
// 35 operations, against seven and 71 with a thread per cell.  The winds'
// positive and negative parts and the reciprocals of G and Gz serve all species
// of the block.  The next level's loads are issued before the level is
// computed.  What bounds it is memory: its accesses' latency and, with species
// groups re-reading the winds, the traffic (1024 x 1024 x 30, 10 FP32 species:
// 3.1 GB it cannot do without, 0.67 ms at the rate of a copy).  Measured
// against a thread per cell: that case 1.20 -> 1.01 ms, 1500 x 1201 x 40, 10
// BF16 and two FP32 species 4.24 -> 2.36 ms, 517 x 389 x 40, 7 species 0.283 ->
// 0.214 ms, 256 x 64 x 20, 12 species 24.4 -> 18.7 us, one species 6.6 -> 7.2.
// NS = 4: two and three species per block take 1.10 and 1.12 ms in the first
// case, six 0.95 but 2.45 in the second; two where the grid is small
// (set_first_blocks), 18.7 us against 26 with four.
constexpr int FCOLS = 62;           // columns a wave writes
constexpr int FWAVES = 4;           // waves of a block
constexpr int FROWS = 2 * FWAVES;   // rows of a block

template <int QK, int NS>
__global__ void __launch_bounds__(64 * FWAVES)
    k_first(const DomDesc *__restrict__ DD, int nd, int fast)
{
    const unsigned blk = xcd_block();
    const DomDesc &D = DD[find_dom_f(DD, nd, blk)];
    unsigned l = blk - D.f0;
    // the species in even groups; those of a tile share its winds in L2
    const int sg = (int)(l % (unsigned)D.fng);
    const int s0 = sg * D.fsb + min(sg, D.fsr), nb = D.fsb + (sg < D.fsr);
    l /= (unsigned)D.fng;
    const int kc = (int)(l % (unsigned)D.fnk), tile = (int)(l / (unsigned)D.fnk);
    const int tx = tile % D.ftx, ty = tile / D.ftx;
    const int nx = D.d.nx, ny = D.d.ny, nz = D.d.nz;
    const int k0 = kc * D.fkch, k1 = min(nz, k0 + D.fkch);
    const int lx = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gi = tx * FCOLS - 1 + lx, j0 = ty * FROWS + 2 * w;  // own rows j0, j0 + 1
    if (j0 >= ny) return;
    const size_t sk = (size_t)nx, sj = (size_t)nx * nz;
    const int x0 = max(0, tx * FCOLS - 1);
    unsigned lane = (unsigned)(min(max(gi, 0), nx - 1) - x0);
    // an offset of which nothing is known: accesses stay scalar plus offset
    auto fresh = [&] { asm("" : "+v"(lane)); };
    size_t rb[4];  // cell (x0, 0) of rows j0 - 1 .. j0 + 2, clamped to the domain
#pragma unroll
    for (int r = 0; r < 4; r++) rb[r] = (size_t)x0 + sj * (size_t)min(max(j0 - 1 + r, 0), ny - 1);
    const bool lane_out = lx >= 1 && lx <= FCOLS && gi < nx;  // gi >= 0 there
    const bool ring_x = gi == 0 || gi == nx - 1;
    SpecPass p[NS];
#pragma unroll
    for (int b = 0; b < NS; b++) {
        p[b] = species(D.pass[0], min(s0 + b, D.nspec - 1));
        if (QK == QK_F32) p[b].kind0 = p[b].kindo = ICAR_ADV_STORE_F32;
    }
    const unsigned tstep = *D.step;

    // four values of a species: the raw bits, and the values (one branch on
    // the kind for the four)
    auto load = [&](const SpecPass &s, const size_t (&c)[4], uint32_t (&r)[4]) {
        fresh();
        if (QK == QK_F32 || s.kind0 == ICAR_ADV_STORE_F32) {
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = ldq<QK_F32>(s.q0, c[e], lane, s.kind0);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = ldq<QK>(s.q0, c[e], lane, s.kind0);
        }
    };
    auto convert = [&](const SpecPass &s, const uint32_t (&r)[4], float (&v)[4]) {
        if (QK == QK_F32 || s.kind0 == ICAR_ADV_STORE_F32) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = __uint_as_float(r[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = cvq<QK>(r[e], s.kind0, s.scale0);
        }
    };
    // the level to come: raw q of rows j0 - 1 and j0 + 2 ([0], [3]) and of the
    // own rows one level further up ([1], [2]), and the winds and divisors
    uint32_t nq[NS][4];
    float nU[2], nV[3], nW[2], nG[2], nZ[2];
    auto fetch = [&](int k) {
        if (k >= k1) return;
        const size_t o = sk * (size_t)k, ou = sk * (size_t)min(k + 1, nz - 1);
        const size_t c[4] = {rb[0] + o, rb[1] + ou, rb[2] + ou, rb[3] + o};
        fresh();
#pragma unroll
        for (int t = 0; t < 2; t++) {
            nU[t] = ld1(D.sf.U, rb[1 + t] + o, lane);
            nW[t] = ld1(D.sf.W, rb[1 + t] + o, lane);
            nG[t] = ld1(D.sf.G, rb[1 + t] + o, lane);
            nZ[t] = ld1(D.sf.Gz, rb[1 + t] + o, lane);
        }
#pragma unroll
        for (int t = 0; t < 3; t++) nV[t] = ld1(D.sf.V, rb[1 + t] + o, lane);
#pragma unroll
        for (int b = 0; b < NS; b++)
            if (b < nb) load(p[b], c, nq[b]);
    };
    // the own rows at level k0 and at the level below it, and the wind between
    uint32_t r0[NS][4];
    float wb[2];
    {
        const size_t o = sk * (size_t)k0, od = sk * (size_t)max(k0 - 1, 0);
        const size_t c[4] = {rb[1] + o, rb[2] + o, rb[1] + od, rb[2] + od};
        fresh();
#pragma unroll
        for (int t = 0; t < 2; t++) wb[t] = ld1(D.sf.W, c[2 + t], lane);
#pragma unroll
        for (int b = 0; b < NS; b++)
            if (b < nb) load(p[b], c, r0[b]);
    }
    fetch(k0);
    float q[NS][2], Fb[NS][2];  // the level's own values, the fluxes through the faces below
#pragma unroll
    for (int b = 0; b < NS; b++) {
        float v[4] = {};
        if (b < nb) convert(p[b], r0[b], v);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            q[b][t] = v[t];
            Fb[b][t] = k0 > 0 ? flux1(v[2 + t], v[t], wb[t]) : 0.0f;
        }
    }
    for (int k = k0; k < k1; k++) {
#pragma unroll
        for (int r = 0; r < 4; r++) asm("" : "+s"(rb[r]));  // no sums of them with every base over the loop
        // this level's winds and values, the next level's on their way
        float U[2], V[3], W[2], G[2], Z[2], qs[NS], qn[NS], qu[NS][2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            U[t] = nU[t];
            W[t] = nW[t];
            G[t] = nG[t];
            Z[t] = nZ[t];
        }
#pragma unroll
        for (int t = 0; t < 3; t++) V[t] = nV[t];
#pragma unroll
        for (int b = 0; b < NS; b++) {
            if (b >= nb) continue;
            float v[4];
            convert(p[b], nq[b], v);
            qs[b] = v[0];
            qn[b] = v[3];
            qu[b][0] = k + 1 < nz ? v[1] : 0.0f;
            qu[b][1] = k + 1 < nz ? v[2] : 0.0f;
        }
        fetch(k + 1);
        // flux1 with the winds' parts formed once for the species of the block
        struct Wind {
            float up, dn;
            __device__ __forceinline__ explicit Wind(float u) : up(u + fabsf(u)), dn(u - fabsf(u)) {}
            __device__ __forceinline__ float flux(float l, float r) const { return (up * l + dn * r) / 2.0f; }
        };
        const Wind wy[3] = {Wind(V[0]), Wind(V[1]), Wind(V[2])};
        float xh[NS][2], xv[NS][2];
#pragma unroll
        for (int b = 0; b < NS; b++) {
            if (b >= nb) continue;
            const float fy[3] = {wy[0].flux(qs[b], q[b][0]), wy[1].flux(q[b][0], q[b][1]),
                                 wy[2].flux(q[b][1], qn[b])};
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const float fl = Wind(U[t]).flux(lane_prev(q[b][t]), q[b][t]), fr = lane_next(fl);
                // the top flux is not upwinded (:96-97)
                const float fz = k > 0 && k == nz - 1 ? q[b][t] * W[t] : Wind(W[t]).flux(q[b][t], qu[b][t]);
                xh[b][t] = (fr - fl) + (fy[t + 1] - fy[t]);  // :86-87
                xv[b][t] = fz - Fb[b][t];                    // :90-94
                Fb[b][t] = fz;
            }
        }
        float v[NS][2];
        // The fast quotients hold for divisors in [2^-30, 2^30] and numerators
        // that are zero or in [2^-96, 2^90]
        auto update = [&](auto fd_c) -> bool {
            constexpr bool F = decltype(fd_c)::value;
            float yG[2] = {}, yZ[2] = {}, big = 0.0f;
            uint32_t key = 0xffffffffu;
            bool in = true;
            if (F) {
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    yG[t] = recip_nr(G[t]);
                    yZ[t] = recip_nr(Z[t]);
                }
                in = vmin3(G[0], G[1], fminf(Z[0], Z[1])) >= 0x1p-30f &&
                     vmax3(G[0], G[1], fmaxf(Z[0], Z[1])) <= 0x1p30f;
            }
#pragma unroll
            for (int b = 0; b < NS; b++) {
                if (b >= nb) continue;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const float x = q[b][t] - fdiv_y<F>(xh[b][t], G[t], yG[t]);
                    v[b][t] = x - fdiv_y<F>(xv[b][t], Z[t], yZ[t]);
                    if (F) {
                        key = min(key, min(nz_key(xh[b][t]), nz_key(xv[b][t])));
                        big = vmax3a(big, xh[b][t], xv[b][t]);
                    }
                }
            }
            return in && key >= ((127u - 96u) << 24) - 1u && big <= 0x1p90f;
        };
        if (!fast || !__all(update(std::integral_constant<bool, true>{})))
            update(std::integral_constant<bool, false>{});
#pragma unroll
        for (int b = 0; b < NS; b++) {
            if (b >= nb) continue;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int j = j0 + t;
                const float r = ring_x || j == 0 || j == ny - 1 ? q[b][t] : v[b][t];  // the ring is copied (:61-63)
                if (lane_out && j < ny) {
                    const size_t c = rb[1 + t] + sk * (size_t)k;
                    fresh();
                    const uint32_t rnd = is_sr(p[b].kindo) ? sr_bits((uint32_t)c + lane, s0 + b, tstep) : 0u;
                    stq<QK>(p[b].out, c, lane, p[b].kindo, p[b].inv_scaleo, r, rnd);
                    if (QK == QK_F32 && D.keep) stq<QK_F32>(D.keep, c, lane, 0, 1.0f, q[b][t], 0u);
                }
                q[b][t] = qu[b][t];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// fused corrective pass
// ---------------------------------------------------------------------------
constexpr int CX = 64;            // staged tile width (one wavefront per row)
constexpr int CH = 2;             // halo
constexpr int CTI = CX - 2 * CH;  // 60 output columns

// A corrective tile of TJ output rows (16 or 8): CY = TJ + 4 staged rows, RW
// output rows per wave.  16 rows recompute fewer halo faces (19 y faces per 16
// rows against 11 per 8), 8 rows give twice the blocks on a small grid, and
// one row per wave (74 registers, six waves per SIMD, against 114 and four)
// the shortest serial work per level; the autotuner times them.  Measured,
// 16 rows x 2 / 8 x 2 / 8 x 1: 1024 x 1024 x 30, 10 FP32 species 3.89 / 3.97 /
// 4.03 ms; 517 x 389 x 40, 7 species 0.89 / 0.83 / 0.82 ms; 256 x 64 x 20, one
// species 23.1 / 18.8 / 17.3 us.  Wave w stages and owns rows 2 + RW w and up;
// the four halo rows are staged by waves 0..3, one each.
template <int TJ, int RW>
struct Tile {
    static constexpr int CY = TJ + 2 * CH;
    static constexpr int NW = TJ / RW;
    static constexpr int CNT = 64 * NW;
    static constexpr int WPE = RW == 2 ? 4 : 6;
    static_assert(NW >= 4, "four waves stage the halo rows");
};

// s = RN(a + b) and its rounding error e, a + b = s + e exactly (Knuth's
// TwoSum; the unit is compiled without contraction)
__device__ __forceinline__ float two_sum(float a, float b, float &e)
{
    const float s = a + b;
    const float bb = s - a;
    e = (a - (s - bb)) + (b - bb);
    return s;
}

// The opt-in compensated form of the update q1 - ((fr-fl) + (fn-fs))/G -
// (Fzt-Fzb)/Gz (upwind_advection, adv_mpdata.f90:86-97): the flux sums and
// the two subtractions carry their rounding errors (TwoSum), the quotients
// their remainders (one FMA each), and the errors enter once, before the
// final rounding; the result is q1 minus the exact divergence of the FP32
// fluxes, rounded about once.  Not the reference's operation order.
__device__ __forceinline__ float divergence_compensated(float q1, float fl, float fr, float fs,
                                                        float fn, float fzt, float fzb, float G,
                                                        float Gz)
{
    float ea, eb, eh, ez, e1, e2;
    const float a = two_sum(fr, -fl, ea);
    const float b = two_sum(fn, -fs, eb);
    const float h = two_sum(a, b, eh);
    const float dh = h / G;
    const float ch = (__builtin_fmaf(-dh, G, h) + ((ea + eb) + eh)) / G;
    const float vz = two_sum(fzt, -fzb, ez);
    const float dz = vz / Gz;
    const float cz = (__builtin_fmaf(-dz, Gz, vz) + ez) / Gz;
    const float t = two_sum(q1, -dh, e1);
    const float u = two_sum(t, -dz, e2);
    return u + ((e1 + e2) - (ch + cz));
}

// A face velocity u limited by the betas of the cells on its positive (p)
// and negative (m) side (adv_mpdata_FCT_core.f90:103-115): u times the
// smallest of 1, the receiving cell's beta_in and the giving cell's beta_out.
// A zero u stays zero whichever pair is taken.
__device__ __forceinline__ float limit_u(float u, bool up, float bi_p, float bo_p, float bi_m,
                                         float bo_m)
{
    return vmin1(up ? bi_p : bi_m, up ? bo_m : bo_p) * u;
}

// Where the corrective kernel takes the three-operation quotient.
//
// Every float is a multiple of the last place of the smallest non-zero float
// around it, so values that are +0 or in [2^lo, 2^hi] have sums and
// differences that are 0 or at least 2^(lo-23) (rounding only coarsens the
// multiples), and the bounds on the numerators and divisors of every quotient
// of a level follow from the range of the staged q1 and q0 alone, once the
// coefficients are bounded (k_coef): each staged level is checked as it is
// staged (two integer extrema per value), and a level's quotients take the
// fast form if the four levels they read are in one of two ranges of 80
// binades.  Then, with eps and 1e-15 in the divisors,
//   - numerators that are sums or differences are 0 or >= 2^-99 (exact
//     remainders need 2^-101), divisors lie in [2^-50, 2^56], quotients are 0
//     or >= 2^(lo-23-hi-20) = 2^-123, normal;
//   - the products in the pseudo-velocities (coefficient times difference or
//     ratio) may be smaller: their smallest non-zero magnitude is tracked
//     (1.5 operations per product) and a wave that meets one below 2^-88
//     computes the phase again with the IEEE division.
// The two ranges: mixing ratios (8e-24 .. 16 per unit) and temperatures or
// number concentrations (1e-14 .. 1.7e10).
struct QRange {
    uint32_t lo, hi;  // bit patterns
};
constexpr QRange QR_SMALL = {(127u - 76u) << 23, (127u + 4u) << 23};
constexpr QRange QR_LARGE = {(127u - 46u) << 23, (127u + 34u) << 23};
constexpr uint32_t KEY_MIN = ((127u - 88u) << 24) - 1u;  // nz_key(2^-88)

// One block marches a (tile, species) column upwards.  Iteration m holds q1
// of levels m-3 .. m in LDS and computes
//   B  the z faces on top of level m-1 and the x/y faces of level m-2
//   -- barrier
//   C  the betas: x within the wave's rows (the neighbours' values come by
//      lane moves, so the x direction is finished here), z within the
//      thread's column, y to LDS; level m+1 is staged
//   -- barrier
//   D  the y fluxes and the divergence of level m-2; level m+2 is prefetched
// What bounds it is VALU issue (a reciprocal takes four slots of a multiply,
// maxima, selects and integer operations two), so the phases do the reference's operations
// and little else: quotients take 6 operations instead of 11 (3 where the
// divisor is shared), each limited x and y face is computed once per wave,
// the bounds use max(q0,q1) and min(q0,q1) staged once per value,
// out-of-domain rows and lanes hold clamped copies and are computed like the
// others (their values reach no output, so no phase masks lanes), levels and
// tiles away from the domain's edges take phases without their tests, and
// every global load is a scalar base plus one 32-bit lane offset.  Two
// barriers per level: the planes a phase writes are those no wave reads
// before the next barrier.  What only its own thread reads stays out of LDS
// (12 planes: four 60 x 8 blocks of four waves fit on a CU, with 15 three).
// Measured per launch: 1024 x 1024 x 30, 10 FP32 species, 5.80 ms with IEEE
// quotients, three barriers and the faces limited once per cell, 4.10 without
// those, 3.89 with 12 planes, scalar bases and the phases without tests; 517
// x 389 x 40, 7 species 1.38, 0.92 and 0.83 ms; 256 x 64 x 20, one species
// 40, 20 and 17 us.
template <bool FCT, int RW, int QK, int TJ>
__global__ void __launch_bounds__((Tile<TJ, RW>::CNT))
    __attribute__((amdgpu_waves_per_eu(Tile<TJ, RW>::WPE, Tile<TJ, RW>::WPE)))
    k_corr(const DomDesc *__restrict__ DD, int nd, int pass, unsigned nwork, int fast)
{
    constexpr int CY = Tile<TJ, RW>::CY;
    // XCD-aware mapping: consecutive work items (the species of one tile)
    // land on the same XCD (blocks are dealt round-robin over 8 XCDs) and
    // share the tile's coefficients in its L2.
    const unsigned nb = gridDim.x;
    const unsigned wi = (blockIdx.x & 7) * (nb >> 3) + (blockIdx.x >> 3);
    if (wi >= nwork) return;
    const DomDesc &D = DD[find_dom_w(DD, nd, wi)];
    const unsigned lw = wi - D.w0;
    const int s = (int)(lw % (unsigned)D.nspec);
    const unsigned tk = lw / (unsigned)D.nspec;
    const int kc = (int)(tk % (unsigned)D.nks);  // column chunk
    const int tile = (int)(tk / (unsigned)D.nks);
    const int tx = tile % D.tiles_x, ty = tile / D.tiles_x;
    const int nx = D.d.nx, ny = D.d.ny, nz = D.d.nz;
    // Levels [k0, k1) of the column are written by this block.  The march
    // starts two levels below k0: the flux through the face under k0 needs
    // the betas of level k0-1, and these the face under it, so with levels
    // k0-2 and up the pipeline holds what a march from the ground would hold
    // when it reaches k0.  The x/y faces below k0 are not computed.
    const int k0 = kc * D.kch;
    const int k1 = min(nz, k0 + D.kch);
    const int m0 = max(0, k0 - 2);
    const size_t sk = (size_t)nx, sj = (size_t)nx * nz;
    const size_t N = sj * ny;
    const int lx = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gi = tx * CTI - CH + lx;
    const int j0 = ty * TJ - CH;  // global row of staged row 0
    const int r0 = 2 + RW * w;    // first owned staged row
    const bool has_x = w < 4;     // this wave stages a halo row as well
    const int rx = w < 2 ? w : TJ + w;  // rows 0, 1, TJ+2, TJ+3

    SpecPass p = species(D.pass[pass - 1], s);
    if (QK == QK_F32) p.kind0 = p.kindo = ICAR_ADV_STORE_F32;  // an FP32-only batch: no 16-bit code
    const bool same = p.q1 == nullptr;
    const unsigned tstep = is_sr(p.kindo) ? *D.step : 0u;
    const bool dom_ok = fast && D.step[1] == 0u;  // coefficients in range (k_coef)
    const float eps = 1e-10f, eps15 = 1e-15f;

    // Global addresses: the row (clamped to the domain), the level and the
    // tile's first column are scalar, the lane's clamped column is one offset
    const int x0 = max(0, tx * CTI - CH);
    unsigned lo = (unsigned)(min(max(gi, 0), nx - 1) - x0);
    // an offset of which nothing is known: its multiples are not kept in
    // registers over the levels, and addresses stay scalar plus offset
    auto fresh = [&] { asm("" : "+v"(lo)); };
    auto row_at = [&](int r) -> size_t {  // cell (x0, 0, row r)
        return (size_t)x0 + sj * (size_t)min(max(j0 + r, 0), ny - 1);
    };
    size_t ra[RW];
#pragma unroll
    for (int t = 0; t < RW; t++) ra[t] = row_at(r0 + t);
    size_t rax = row_at(has_x ? rx : r0);
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) const f4 gcf4;
    auto ld1 = [&](const float *b, size_t c) -> float { return icaradv::ld1(b, c, lo); };
    auto ld4 = [&](const float *b, size_t c) -> f4 {
        return *(gcf4 *)((gcchar *)(gcfloat *)(b + 4 * c) + lo * 16u);
    };
    auto ldq = [&](size_t c) -> uint32_t { return icaradv::ldq<QK>(p.q0, c, lo, p.kind0); };
    auto cvq = [&](uint32_t b) -> float { return icaradv::cvq<QK>(b, p.kind0, p.scale0); };

    // LDS planes of CY rows of 64 floats (a wave reads one row, lane i at
    // word i, so no bank conflicts)
    constexpr int PL = CY * CX;
    __shared__ float lds[CX + 12 * PL];
    __shared__ int out_of[4][2];  // level & 3: a value outside QR_SMALL / QR_LARGE
    float *const Q = lds + CX;    // q1, ring by level & 3 (CX floats below it: lane -1 of row 0)
    float *const MX = Q + 4 * PL;   // max(q0, q1), ring by level & 1
    float *const MN = MX + 2 * PL;  // min(q0, q1)
    float *const VU = MN + 2 * PL;  // y face south of a row: its velocity
    float *const VF = VU + PL;      //   and its donor flux
    float *const BI = VF + PL, *const BO = BI + PL;  // y betas

    const int own = r0 * CX + lx, ext = rx * CX + lx;
    const bool lane_out = lx >= CH && lx < CX - CH && gi < nx;  // gi >= 0 there
    const int gj0 = j0 + r0;
    const bool edge_x = tx == 0 || tx == D.tiles_x - 1 || tx * CTI + CTI + 1 >= nx - 1;
    const bool at_w = gi == 0, at_e = gi == nx - 1;
    // no cell whose betas are used is in the domain's ring of rows or columns
    const bool inner = !edge_x && j0 >= 0 && j0 + TJ + 2 < ny - 1;

    // z pipeline of the two owned columns
    float wu2[RW], wu1[RW], fz2[RW], fz1[RW];  // unlimited w and its flux on faces m-2, m-1
    float bzi[RW], bzo[RW];                  // betas of the cell below the current one
    float Fzp[RW];                          // flux on the face below the output level
#pragma unroll
    for (int t = 0; t < RW; t++) {
        wu2[t] = wu1[t] = fz2[t] = fz1[t] = 0.0f;
        bzi[t] = bzo[t] = 1.0f;
        Fzp[t] = 0.0f;
    }

    uint32_t n0[RW + 1];  // the next level to stage: raw q0 and q1
    float n1[RW + 1];
    float bx[RW + 1], bn[RW + 1];  // max(q0, q1) and min(q0, q1) of the level staged last
    auto prefetch = [&](int m) {
        if (m < nz) {
            fresh();
            const size_t c = sk * (size_t)m;
#pragma unroll
            for (int t = 0; t < RW; t++) n0[t] = ldq(ra[t] + c);
            if (has_x) {
                fresh();
                n0[RW] = ldq(rax + c);
            }
            if (!same) {
                fresh();
#pragma unroll
                for (int t = 0; t < RW; t++) n1[t] = ld1(p.q1, ra[t] + c);
                if (has_x) {
                    fresh();
                    n1[RW] = ld1(p.q1, rax + c);
                }
            }
        }
    };
    // level m into its q1 plane
    auto stage = [&](int m) {
        if (m >= nz) return;
        float *const q = Q + (m & 3) * PL;
        uint32_t klo = 0xffffffffu, khi = 0u;
#pragma unroll
        for (int r = 0; r < RW + 1; r++) {
            if (r == RW && !has_x) continue;
            const float a = cvq(n0[r]), b = same ? a : n1[r];
            q[r < RW ? own + CX * r : ext] = b;
            // the extremes of both fields, as unsigned bit patterns: -0 and
            // negative values, infinities and NaN compare above every range,
            // and +0 (minus 1) never counts as small
            klo = min(klo, min(__float_as_uint(a) - 1u, __float_as_uint(b) - 1u));
            khi = max(khi, max(__float_as_uint(a), __float_as_uint(b)));
        }
        const bool os = klo < QR_SMALL.lo - 1u || khi > QR_SMALL.hi;
        const bool ol = klo < QR_LARGE.lo - 1u || khi > QR_LARGE.hi;
        if (__any(os)) out_of[m & 3][0] = 1;
        if (__any(ol)) out_of[m & 3][1] = 1;
    };
    // The maxima and minima of the bounds of the level staged last; they stay
    // in registers for a level, where only this thread needs them (the z
    // direction), and then go to their planes, which so hold two levels.
    auto bounds = [&](int m) {
        if (!FCT || m >= nz) return;
#pragma unroll
        for (int r = 0; r < RW + 1; r++) {
            if (r == RW && !has_x) continue;
            const float a = cvq(n0[r]), b = same ? a : n1[r];
            bx[r] = vmax(a, b);
            bn[r] = vmin(a, b);
        }
    };
    auto put_bounds = [&](int m) {
        if (!FCT || m >= nz) return;
        const int o = (m & 1) * PL;
#pragma unroll
        for (int r = 0; r < RW + 1; r++) {
            if (r == RW && !has_x) continue;
            const int c = o + (r < RW ? own + CX * r : ext);
            MX[c] = bx[r];
            MN[c] = bn[r];
        }
    };

    f4 kx[RW], kz[RW], ky[RW + 1];
    float kd[RW];
    // The coefficients of iteration m; a level out of range reads the nearest
    // one (its values are not used)
    auto load_coef = [&](int m) {
        fresh();
        const size_t c2 = sk * (size_t)min(max(m - 2, 0), nz - 1);
        const size_t c1 = sk * (size_t)max(0, min(m - 1, nz - 2));
        const float *gx = D.coef, *gy = gx + 4 * N, *gz = gx + 8 * N;
#pragma unroll
        for (int t = 0; t < RW; t++) {
            kz[t] = ld4(gz, ra[t] + c1);
            kd[t] = ld1(D.f.dz, ra[t] + c1);
        }
#pragma unroll
        for (int t = 0; t < RW; t++) kx[t] = ld4(gx, ra[t] + c2);
#pragma unroll
        for (int t = 0; t < RW; t++) ky[t] = ld4(gy, ra[t] + c2);
        if (has_x) {
            fresh();
            ky[RW] = ld4(gy, rax + c2);
        }
    };

    if (threadIdx.x < CX) {
        lds[threadIdx.x] = 0.0f;
        if (threadIdx.x < 8) out_of[threadIdx.x >> 1][threadIdx.x & 1] = 0;
    }
    __syncthreads();
    prefetch(m0);
    stage(m0);
    bounds(m0);
    prefetch(m0 + 1);
    __syncthreads();

    constexpr std::integral_constant<bool, true> yes;
    constexpr std::integral_constant<bool, false> no;
    int hs = 0, hl = 0;  // out_of of levels m, m-1, m-2, m-3 in bits 0..3
    for (int m = m0; m <= k1 + 1; m++) {
#pragma unroll
        for (int t = 0; t < RW; t++) asm("" : "+s"(ra[t]));
        asm("" : "+s"(rax));
        const int L1 = m - 1, L2 = m - 2;
        const bool xy = L2 >= k0;  // (L2 < k1 by the loop's end)
        const bool zf = L1 >= m0 && L1 <= nz - 1;
        const bool mid = L2 >= max(k0, 1) && m < nz;  // no phase meets the ground or the top
        const float *const qm = Q + (m & 3) * PL + own;         // level m
        const float *const qu = Q + ((m + 3) & 3) * PL + own;   // level m-1 = L1 = L2+1
        const float *const qc = Q + ((m + 2) & 3) * PL + own;   // level m-2 = L2
        const float *const qd = Q + ((m + 1) & 3) * PL + own;   // level m-3 = L2-1
        load_coef(m);
        float kg[RW], kgz[RW];
        if (xy) {
            const size_t c2 = sk * (size_t)L2;
            fresh();
#pragma unroll
            for (int t = 0; t < RW; t++) {
                kg[t] = ld1(D.sf.G, ra[t] + c2);
                kgz[t] = ld1(D.sf.Gz, ra[t] + c2);
            }
        }
        hs = (hs << 1) & 15;
        hl = (hl << 1) & 15;
        if (m < nz) {
            hs |= __builtin_amdgcn_readfirstlane(out_of[m & 3][0]);
            hl |= __builtin_amdgcn_readfirstlane(out_of[m & 3][1]);
        }
        const bool ok = dom_ok && (hs == 0 || hl == 0);

        // ---------------- (B) unlimited pseudo-velocities (mpdata_fluxes)
        // A phase computed again writes the same places.
        float zw[RW] = {}, zq[RW] = {}, xu[RW], xf[RW], yu[RW + 1], yf[RW + 1];
        auto phase_b = [&](auto fd_c, auto mid_c) -> uint32_t {
            constexpr bool F = decltype(fd_c)::value, M = decltype(mid_c)::value;
            uint32_t key = 0xffffffffu;
            // a face's value: its first term and two cross terms (the second
            // where the face has levels on both sides)
            auto face = [&](float l, float r, f4 k, float d1, float s1, bool two, float d2,
                            float s2) -> float {
                const float x = k.x * (r - l);
                float val = fdiv<F>(x, r + l + eps);
                const float y = F ? recip_nr(k.w) : 0.0f;
                const float x1 = k.y * fdiv<F>(d1, s1 + eps);
                val = val - fdiv_y<F>(x1, k.w, y);
                if (F) key = min(key, min(nz_key(x), nz_key(x1)));
                if (two) {
                    const float x2 = k.z * fdiv<F>(d2, s2 + eps);
                    val = val - fdiv_y<F>(x2, k.w, y);
                    if (F) key = min(key, nz_key(x2));
                }
                return val;
            };
            // z face on top of level L1 for the owned columns (:211-246, :380)
            if (M || zf) {
                if (M || L1 <= nz - 2) {
#pragma unroll
                    for (int t = 0; t < RW; t++) {
                        const float *a = qu + CX * t, *b = qm + CX * t;  // levels k and k+1
                        const float l = a[0], r = b[0];
                        // WxU (:227-233), WxV (:238-245)
                        const float v = face(l, r, kz[t],
                                             b[1] - a[-1] + a[1] - b[-1], a[1] + b[1] + a[-1] + b[-1], true,
                                             b[CX] - a[-CX] + a[CX] - b[-CX],
                                             a[CX] + b[-CX] + b[CX] + a[-CX]);
                        zw[t] = v * 0.5f * kd[t];
                        zq[t] = flux1(l, r, zw[t]);
                    }
                }
            }
            if (M || xy) {
                const bool kin = M || (L2 >= 1 && L2 <= nz - 2);
                // x faces left of the owned rows' cells (:131-165, :378)
#pragma unroll
                for (int t = 0; t < RW; t++) {
                    const float *c = qc + CX * t, *u = qu + CX * t, *d = qd + CX * t;
                    const float l = c[-1], r = c[0];
                    // UxV (:145-152), UxW (:157-164)
                    float d2 = 0.0f, s2 = 0.0f;
                    if (kin) {
                        d2 = u[0] - d[0] + u[-1] - d[-1];
                        s2 = u[0] + d[0] + u[-1] + d[-1];
                    }
                    const float v = face(l, r, kx[t],
                                         c[CX] - c[-CX] + c[CX - 1] - c[-CX - 1],
                                         c[CX] + c[-CX] + c[CX - 1] + c[-CX - 1], kin, d2, s2);
                    xu[t] = v * 0.5f;
                    xf[t] = flux1(l, r, xu[t]);
                }
                // y faces south of the owned rows and the halo rows 1, TJ+2
                // and TJ+3 (:169-205, :379)
#pragma unroll
                for (int t = 0; t < RW + 1; t++) {
                    if (t == RW && (!has_x || w == 0)) continue;
                    const int o = t < RW ? CX * t : ext - own;
                    const float *c = qc + o, *u = qu + o, *d = qd + o;
                    const float l = c[-CX], r = c[0];
                    // VxU (:186-192), VxW (:197-204)
                    float d2 = 0.0f, s2 = 0.0f;
                    if (kin) {
                        d2 = u[-CX] - d[0] + u[0] - d[-CX];
                        s2 = u[-CX] + d[0] + u[0] + d[-CX];
                    }
                    const float v = face(l, r, ky[t],
                                         c[1 - CX] - c[-1] + c[1] - c[-CX - 1],
                                         c[1] + c[1 - CX] + c[-1] + c[-CX - 1], kin, d2, s2);
                    yu[t] = v * 0.5f;
                    yf[t] = flux1(l, r, yu[t]);
                    VU[own + o] = yu[t];
                    VF[own + o] = yf[t];
                }
            }
            return key;
        };
        {
            bool ieee = true;
            if (ok) {
                const uint32_t key = mid ? phase_b(yes, yes) : phase_b(yes, no);
                ieee = __any(key < KEY_MIN);
            }
            if (ieee) phase_b(no, no);
        }
        if (zf) {
#pragma unroll
            for (int t = 0; t < RW; t++) {
                wu2[t] = wu1[t];
                fz2[t] = fz1[t];
                wu1[t] = zw[t];
                fz1[t] = zq[t];
            }
        }
        __syncthreads();

        // ---------------- (C) FCT: per-cell betas (adv_mpdata_FCT_core.f90:47-116)
        float Fzc[RW] = {};  // flux on top of level L2
        float Fxl[RW], Fxr[RW];  // limited fluxes of the x faces
        const int o2 = (L2 & 1) * PL, o1 = (L1 & 1) * PL;
        // the y face south of the row north of the owned ones: its velocity, or
        // without FCT its flux (read before the barrier: the next level's
        // phase B overwrites the plane)
        float yn = 0.0f;
        if (FCT) {
            auto phase_c = [&](auto fd_c, auto mid_c) {
                constexpr bool F = decltype(fd_c)::value, M = decltype(mid_c)::value;
                // the betas of a cell from its bounds and the fluxes of its
                // two faces in one direction
                auto betas = [&](float q, float hi, float low, float fin, float fout, float &bi,
                                 float &bo) {
                    bi = fdiv<F>(hi - q, fin + eps15);
                    bo = fdiv<F>(q - low, fout + eps15);
                };
                if (M || xy) {
#pragma unroll
                    for (int t = 0; t < RW; t++) {
                        const int c = o2 + own + CX * t;
                        const float q = qc[CX * t], ql = qc[CX * t - 1];
                        float xw = MX[c - 1], xc = MX[c], xe = MX[c + 1];
                        float nw = MN[c - 1], nc = MN[c], ne = MN[c + 1];
                        const float fl = xf[t], fr = lane_next(fl);
                        float fin = vpos(fl) - vneg(fr), fout = vpos(fr) - vneg(fl);
                        if (!M && edge_x) {  // the row's end cells: :50-55, :62-68, :79-83, :95-99
                            xw = at_w ? xc : xw;
                            nw = at_w ? nc : nw;
                            xc = at_e ? q : xc;
                            nc = at_e ? q : nc;
                            xe = at_e ? q : xe;
                            ne = at_e ? q : ne;
                            fin = at_w || at_e ? 0.0f : fin;
                            fout = at_w || at_e ? 0.0f : fout;
                        }
                        float bi, bo;
                        betas(q, vmax3(xw, xc, xe), vmin3(nw, nc, ne), fin, fout, bi, bo);
                        const float bil = lane_prev(bi), bol = lane_prev(bo);
                        const float u = limit_u(xu[t], xu[t] > 0.0f, bi, bo, bil, bol);
                        Fxl[t] = flux1(ql, q, u);
                        Fxr[t] = lane_next(Fxl[t]);
                    }
                    // y cells on the owned rows and the halo rows 1 and TJ+2
#pragma unroll
                    for (int t = 0; t < RW + 1; t++) {
                        if (t == RW && !(w == 1 || w == 2)) continue;
                        const int o = t < RW ? CX * t : ext - own;
                        const int c = o2 + own + o, gj = t < RW ? gj0 + t : j0 + rx;
                        const float q = qc[o];
                        float hi, low, fin, fout;
                        if (!M && gj <= 0) {
                            hi = vmax(MX[c], MX[c + CX]);
                            low = vmin(MN[c], MN[c + CX]);
                            fin = fout = 0.0f;
                        } else if (!M && gj >= ny - 1) {
                            hi = vmax(MX[c - CX], q);
                            low = vmin(MN[c - CX], q);
                            fin = fout = 0.0f;
                        } else {
                            hi = vmax3(MX[c - CX], MX[c], MX[c + CX]);
                            low = vmin3(MN[c - CX], MN[c], MN[c + CX]);
                            const float fs = yf[t], fn = VF[own + o + CX];
                            fin = vpos(fs) - vneg(fn);
                            fout = vpos(fn) - vneg(fs);
                        }
                        float bi, bo;
                        betas(q, hi, low, fin, fout, bi, bo);
                        BI[own + o] = bi;
                        BO[own + o] = bo;
                    }
                }
                // z: betas of cell L1 of each owned column, then the limited
                // velocity and flux on the face between L2 and L1 (flux_is_w ends)
                if (M || zf) {
#pragma unroll
                    for (int t = 0; t < RW; t++) {
                        const int c = own + CX * t;
                        const float q = qu[CX * t];
                        float hi, low, fin, fout;
                        if (!M && L1 == 0) {
                            hi = vmax(MX[o1 + c], bx[t]);
                            low = vmin(MN[o1 + c], bn[t]);
                            fin = 0.0f - vneg(fz1[t]);
                            fout = vpos(fz1[t]);
                        } else if (!M && L1 == nz - 1) {
                            hi = vmax(MX[o2 + c], q);
                            low = vmin(MN[o2 + c], q);
                            fin = vpos(fz2[t]) - vneg(fz2[t]);
                            fout = fin;
                        } else {
                            hi = vmax3(MX[o2 + c], MX[o1 + c], bx[t]);
                            low = vmin3(MN[o2 + c], MN[o1 + c], bn[t]);
                            fin = vpos(fz2[t]) - vneg(fz1[t]);
                            fout = vpos(fz1[t]) - vneg(fz2[t]);
                        }
                        float bi, bo;
                        betas(q, hi, low, fin, fout, bi, bo);
                        if (M || L2 >= m0) {
                            const float u = limit_u(wu2[t], wu2[t] > 0.0f, bi, bo, bzi[t], bzo[t]);
                            Fzc[t] = flux1(qc[CX * t], q, u);
                        }
                        bzi[t] = bi;
                        bzo[t] = bo;
                    }
                }
            };
            if (!ok) phase_c(no, no);
            else if (mid && inner) phase_c(yes, yes);
            else phase_c(yes, no);
            yn = VU[own + RW * CX];
        } else {
            yn = VF[own + RW * CX];
#pragma unroll
            for (int t = 0; t < RW; t++) {
                if (L2 >= m0 && L2 <= nz - 2) Fzc[t] = fz2[t];
                if (xy) {
                    Fxl[t] = xf[t];
                    Fxr[t] = lane_next(xf[t]);
                }
            }
        }
        stage(m + 1);
        __syncthreads();

        // ---------------- (D) flux divergence on level L2 (upwind_advection
        // :86-97) with the limited velocities of the cell's four side faces
        if (threadIdx.x < 2) out_of[(m + 2) & 3][threadIdx.x] = 0;
        put_bounds(m);
        bounds(m + 1);
        prefetch(m + 2);
        if (xy) {
            // the y faces south of the owned rows and of the row north of them
            float Fy[RW + 1];
            if (FCT) {
#pragma unroll
                for (int t = 0; t < RW + 1; t++) {
                    const int c = own + CX * t;
                    const float v = t < RW ? yu[t] : yn;
                    const float u = limit_u(v, v > 0.0f, BI[c], BO[c], BI[c - CX], BO[c - CX]);
                    Fy[t] = flux1(qc[CX * (t - 1)], qc[CX * t], u);
                }
            } else {
#pragma unroll
                for (int t = 0; t < RW; t++) Fy[t] = yf[t];
                Fy[RW] = yn;
            }
#pragma unroll
            for (int t = 0; t < RW; t++) {
                const int gj = gj0 + t;
                float q = qc[CX * t];
                // the top flux is the value times a velocity of 0 (:96-97): a zero of
                // its sign, and NaN for what is not finite.  Selected here for
                // every level; a branch at the top cost 1.2% of a run of 256 x
                // 64 x 20, one species (562 -> 569 us), this nothing
                const float fzt = L2 == nz - 1 ? q * 0.0f : Fzc[t];
                if (gj > 0 && gj < ny - 1) {  // the ring keeps its values
                    float v;
                    if (D.compensated) {
                        v = divergence_compensated(q, Fxl[t], Fxr[t], Fy[t], Fy[t + 1], fzt, Fzp[t],
                                                   kg[t], kgz[t]);
                    } else {
                        v = q - ((Fxr[t] - Fxl[t]) + (Fy[t + 1] - Fy[t])) / kg[t];
                        v = v - (fzt - Fzp[t]) / kgz[t];
                    }
                    q = at_w || at_e ? q : v;
                }
                if (lane_out && gj < ny) {  // gj >= 0: owned rows start at the tile's first
                    const size_t c = ra[t] + sk * (size_t)L2;
                    fresh();
                    const uint32_t rnd = is_sr(p.kindo) ? sr_bits((uint32_t)c + lo, s, tstep) : 0u;
                    stq<QK>(p.out, c, lo, p.kindo, p.inv_scaleo, q, rnd);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < RW; t++) Fzp[t] = Fzc[t];
    }
}

// The same ring conditions for every species of every domain of a batch, one
// launch over a table of (domain, species) entries with the species' current
// buffer; a block row per entry.
struct BcEntry {
    Dims d;
    void *q;
    int esz;  // bytes per element: 4 (FP32) or 2 (16-bit kinds)
};

__global__ void __launch_bounds__(256)
    k_bc_all(const BcEntry *__restrict__ tab, int bc_x, int bc_y)
{
    const BcEntry e = tab[blockIdx.y];
    const unsigned t = blockIdx.x * 256u + threadIdx.x;
    if (t >= ring_x_threads(e.d, bc_x) + ring_y_threads(e.d, bc_y)) return;
    if (e.esz == 4) ring_cells(static_cast<uint32_t *>(e.q), e.d, t, bc_x, bc_y);
    else ring_cells(static_cast<uint16_t *>(e.q), e.d, t, bc_x, bc_y);
}

unsigned grid_for(size_t n)
{
    size_t b = (n + 255) / 256;
    if (b > 16384) b = 16384;
    return (unsigned)(b < 1 ? 1 : b);
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct FastState {
    Dims d{};
    size_t N = 0;
    std::string err;
    std::vector<FastSpecies> sp;         // home buffers as bound
    std::vector<void *> alt;             // second home buffer per species
    int cur = 0;                         // which home holds the current state
    int gen = 0;                         // bumped whenever the species buffers change
    float *s1 = nullptr, *s2 = nullptr;  // FP32 scratch, nspec * N each
    float *coef = nullptr;               // NCOEF values per cell (float4 groups)
    SpecPass *d_tab = nullptr;           // [2 parities][passes][nspec]
    int tab_order = -1;
    size_t tab_cap = 0;
    unsigned *d_step = nullptr;          // DomDesc::step
};

struct FastBatch {
    std::vector<FastDomain> doms;
    std::vector<int> gens;
    int order = 0, fct = 0;
    DomDesc *d_desc = nullptr;           // [2 parities][n]
    std::vector<DomDesc> h_desc[2];
    std::vector<float> dts;              // dt values in the device tables
    unsigned total_cb = 0, total_fb = 0, total_work = 0;
    int fns = 4;         // most species of a block of the donor-cell kernel
    double cells = 0, cell_species = 0;  // for the algorithmic byte counts
    int corr_cfg = 3;    // corrective kernel's tile (launch_corr_t)
    int tj = 16;         // output rows per corrective tile (tile_rows(corr_cfg))
    int nks = 1;         // requested column chunks along k
    bool tuned = false;  // launch configuration chosen (autotuned or fixed by the environment)
    bool dirty = true;   // device tables out of date
    bool has_sr = false; // a species is stored with stochastic rounding
    BcEntry *d_bc = nullptr;  // ring-condition table: [2 parities][n_bc] (fast_batch_bc)
    int n_bc = 0;
    bool q16 = false;    // a species is stored in 16 bits
    bool f16 = false;    // a species is stored in FP16 (kernels for any kind)
};

namespace {

size_t kind_bytes(int kind) { return kind == ICAR_ADV_STORE_F32 ? 4 : 2; }

void free_species_buffers(FastState *st)
{
    for (void *p : st->alt) (void)hipFree(p);
    st->alt.clear();
    (void)hipFree(st->s1);
    (void)hipFree(st->s2);
    st->s1 = st->s2 = nullptr;
}

void *home(FastState *st, int s, int which)
{
    return which == 0 ? st->sp[s].dev : st->alt[s];
}

// Per-pass species tables of one domain for both home parities.
int build_tables(FastState *st, int order)
{
    const int S = (int)st->sp.size();
    const int P = order < 1 ? 1 : order;
    const size_t need = (size_t)2 * P * S;
    // FP32 buffers of the intermediate passes: s1 from order 2 on, s2 from
    // order 3 on (at order 1 the donor-cell pass writes the result directly)
    if (P >= 2 && !st->s1 && hipMalloc(&st->s1, (size_t)S * st->N * sizeof(float)) != hipSuccess) {
        st->s1 = nullptr;
        st->err = "hipMalloc of the FP32 pass buffer failed";
        return ICAR_ADV_ENOMEM;
    }
    if (P >= 3 && !st->s2 && hipMalloc(&st->s2, (size_t)S * st->N * sizeof(float)) != hipSuccess) {
        st->s2 = nullptr;
        st->err = "hipMalloc of the second FP32 pass buffer failed";
        return ICAR_ADV_ENOMEM;
    }
    if (need > st->tab_cap) {
        (void)hipFree(st->d_tab);
        st->d_tab = nullptr;
        if (hipMalloc(&st->d_tab, need * sizeof(SpecPass)) != hipSuccess) {
            st->err = "hipMalloc of the species pass tables failed";
            st->tab_cap = 0;
            return ICAR_ADV_ENOMEM;
        }
        st->tab_cap = need;
    }
    std::vector<SpecPass> h(need);
    for (int par = 0; par < 2; par++)
        for (int pass = 1; pass <= P; pass++)
            for (int s = 0; s < S; s++) {
                const FastSpecies &f = st->sp[s];
                const float sc = ldexpf(1.0f, f.pow2), isc = ldexpf(1.0f, -f.pow2);
                float *sa = st->s1 ? st->s1 + (size_t)s * st->N : nullptr;
                float *sb = st->s2 ? st->s2 + (size_t)s * st->N : nullptr;
                SpecPass e{};
                void *hcur = home(st, s, par), *hoth = home(st, s, 1 - par);
                if (pass == 1) {  // q0 = home
                    e.q0 = hcur, e.kind0 = f.storage, e.scale0 = sc, e.q1 = nullptr;
                } else if (pass == 2) {  // q0 = home, q1 = first pass
                    e.q0 = hcur, e.kind0 = f.storage, e.scale0 = sc, e.q1 = sa;
                } else {  // q0 = q1 = previous pass (adv_mpdata.f90:388-397)
                    e.q0 = (pass % 2 == 1) ? sb : sa;
                    e.kind0 = ICAR_ADV_STORE_F32, e.scale0 = 1.0f, e.q1 = nullptr;
                }
                if (pass == P) {  // home is not read after pass 2
                    e.out = (P <= 2) ? hoth : hcur;
                    e.kindo = f.storage, e.inv_scaleo = isc;
                } else {
                    e.out = (pass % 2 == 1) ? sa : sb;
                    e.kindo = ICAR_ADV_STORE_F32, e.inv_scaleo = 1.0f;
                }
                h[((size_t)par * P + (pass - 1)) * S + s] = e;
            }
    if (hipMemcpy(st->d_tab, h.data(), need * sizeof(SpecPass), hipMemcpyHostToDevice) !=
        hipSuccess) {
        st->err = "upload of the species pass tables failed";
        return ICAR_ADV_ENOMEM;
    }
    st->tab_order = order;
    return 0;
}

unsigned cell_blocks(const Dims &d)
{
    return (unsigned)((d.nx + 63) / 64) * (unsigned)d.nz * (unsigned)((d.ny + 3) / 4);
}

}  // namespace

FastState *fast_create(Dims d)
{
    FastState *st = new FastState();
    st->d = d;
    st->N = (size_t)d.nx * d.ny * d.nz;
    if (hipMalloc(&st->coef, (size_t)NCOEF * st->N * sizeof(float)) != hipSuccess ||
        hipMalloc(&st->d_step, 2 * sizeof(unsigned)) != hipSuccess ||
        hipMemset(st->d_step, 0, 2 * sizeof(unsigned)) != hipSuccess) {
        fast_destroy(st);
        return nullptr;
    }
    return st;
}

void fast_destroy(FastState *st)
{
    if (!st) return;
    free_species_buffers(st);
    (void)hipFree(st->coef);
    (void)hipFree(st->d_tab);
    (void)hipFree(st->d_step);
    delete st;
}

int fast_set_species(FastState *st, const FastSpecies *sp, int n, hipStream_t stream)
{
    // At mpdata_order <= 2 the steps alternate between the two home buffers.
    // When the current state sits in the second buffer, a species that keeps
    // its home buffer (same buffer, same storage) gets its current values
    // copied home first, so that binding another species leaves it as it was.
    if (st->cur == 1) {
        for (int s = 0; s < n; s++)
            for (size_t o = 0; o < st->sp.size() && o < st->alt.size(); o++)
                if (st->sp[o].dev == sp[s].dev && st->sp[o].storage == sp[s].storage &&
                    st->alt[o]) {
                    if (hipMemcpyAsync(sp[s].dev, st->alt[o],
                                       st->N * kind_bytes(sp[s].storage), hipMemcpyDeviceToDevice,
                                       stream) != hipSuccess) {
                        st->err = "copy of a species' current state to its home buffer failed";
                        return ICAR_ADV_ENOMEM;
                    }
                    break;
                }
        if (hipStreamSynchronize(stream) != hipSuccess) {
            st->err = "copy of the species' current states to their home buffers failed";
            return ICAR_ADV_ENOMEM;
        }
    }
    free_species_buffers(st);
    st->sp.assign(sp, sp + n);
    st->cur = 0;
    st->tab_order = -1;
    st->gen++;
    if (n == 0) return 0;
    st->alt.assign(n, nullptr);
    for (int s = 0; s < n; s++)
        if (hipMalloc(&st->alt[s], st->N * kind_bytes(sp[s].storage) + 64) != hipSuccess) {
            st->err = "hipMalloc of a species buffer failed";
            return ICAR_ADV_ENOMEM;
        }
    return 0;  // the FP32 pass buffers follow the order (build_tables)
}

void *fast_species_ptr(FastState *st, int s)
{
    if (!st || s < 0 || s >= (int)st->sp.size()) return nullptr;
    return home(st, s, st->cur);
}

int fast_parity(FastState *st) { return st ? st->cur : 0; }

void fast_set_parity(FastState *st, int parity)
{
    if (st) st->cur = parity & 1;
}

const char *fast_error(FastState *st) { return st ? st->err.c_str() : "no fused state"; }

namespace {

constexpr int MIN_CHUNK = 4;  // levels per column chunk at least

// Column chunks of every domain for about nks chunks per column, and the
// work-item layout (tile, chunk, species) that follows from them.
void set_ksplit(FastBatch *b, int nks)
{
    b->nks = nks < 1 ? 1 : nks;
    unsigned w = 0;
    for (size_t k = 0; k < b->doms.size(); k++) {
        const Dims &d = b->doms[k].st->d;
        int kch = (d.nz + b->nks - 1) / b->nks;
        if (kch < MIN_CHUNK) kch = MIN_CHUNK;
        if (kch > d.nz) kch = d.nz;
        const int chunks = (d.nz + kch - 1) / kch;
        const int tiles = ((d.nx + CTI - 1) / CTI) * ((d.ny + b->tj - 1) / b->tj);
        for (int par = 0; par < 2; par++) {
            DomDesc &E = b->h_desc[par][k];
            E.w0 = w;
            E.nks = chunks;
            E.kch = kch;
        }
        w += (unsigned)(tiles * chunks * (int)b->doms[k].st->sp.size());
    }
    b->total_work = w;
    b->dirty = true;
}

// The copies are not ordered with the work on s, which may still read the
// tables: it ends first.
int upload_tables(FastBatch *b, hipStream_t s, std::string *err)
{
    const size_t n = b->doms.size();
    if (hipStreamSynchronize(s) != hipSuccess) {
        *err = "a previous step failed";
        return ICAR_ADV_EINVAL;
    }
    for (int par = 0; par < 2; par++)
        if (hipMemcpy(b->d_desc + (size_t)par * n, b->h_desc[par].data(), n * sizeof(DomDesc),
                      hipMemcpyHostToDevice) != hipSuccess) {
            *err = "upload of the domain table failed";
            return ICAR_ADV_ENOMEM;
        }
    b->dirty = false;
    return 0;
}

// corr_cfg: bit 2 -> 8 tile rows (16 otherwise); bit 0 -> two rows per wave, or,
// clear and with 8 tile rows, one; bit 1 has no effect
template <bool FCT, int QK>
void launch_corr_t(unsigned nb, hipStream_t s, const DomDesc *D, int n, int pass, unsigned nw,
                   int cfg, int fast)
{
    auto go = [&](auto rw, auto tj) {
        hipLaunchKernelGGL((k_corr<FCT, rw.value, QK, tj.value>), dim3(nb),
                           dim3(Tile<tj.value, rw.value>::CNT), 0, s, D, n, pass, nw, fast);
    };
    constexpr std::integral_constant<int, 1> one;
    constexpr std::integral_constant<int, 2> two;
    if (!(cfg & 4)) go(two, std::integral_constant<int, 16>{});
    else if (cfg & 1) go(two, std::integral_constant<int, 8>{});
    else go(one, std::integral_constant<int, 8>{});
}

// the kernels' storage class for a batch: FP32 only, FP32 and BF16, or any kind
int storage_class(const FastBatch *b)
{
    return !b->q16 ? QK_F32 : b->f16 ? QK_ANY : QK_BF16;
}

template <bool FCT>
void launch_corr_q(const FastBatch *b, unsigned nb, hipStream_t s, const DomDesc *D, int n,
                   int pass, unsigned nw, int cfg, int fast)
{
    switch (storage_class(b)) {
    case QK_F32: launch_corr_t<FCT, QK_F32>(nb, s, D, n, pass, nw, cfg, fast); break;
    case QK_BF16: launch_corr_t<FCT, QK_BF16>(nb, s, D, n, pass, nw, cfg, fast); break;
    default: launch_corr_t<FCT, QK_ANY>(nb, s, D, n, pass, nw, cfg, fast); break;
    }
}

int tile_rows(int cfg) { return (cfg & 4) ? 8 : 16; }

// ICAR_ADV_FAST_DIV=0 makes the donor-cell and corrective kernels divide by the
// IEEE sequence throughout (the same results)
int fast_division()
{
    static const int on = [] {
        const char *e = getenv("ICAR_ADV_FAST_DIV");
        return e && *e ? atoi(e) != 0 : 1;
    }();
    return on;
}

void launch_corr(const FastBatch *b, hipStream_t s, const DomDesc *D, int n, int pass, int cfg)
{
    const unsigned nw = b->total_work;
    const unsigned nb = (nw + 7) / 8 * 8;
    const int fast = fast_division();
    if (b->fct) launch_corr_q<true>(b, nb, s, D, n, pass, nw, cfg, fast);
    else launch_corr_q<false>(b, nb, s, D, n, pass, nw, cfg, fast);
}

// Tuned configurations by batch shape, shared by every batch of the process.
std::mutex g_tune_mu;
std::map<std::string, std::pair<int, int>> g_tuned;

// The donor-cell kernel's blocks: columns of four species where those fill the
// GPU, else of two species and in as many level chunks as it takes (a chunk
// loads one level more).
void set_first_blocks(FastBatch *b)
{
    constexpr int FILL = 1024;  // four blocks per CU
    auto groups = [&](size_t k) { return ((int)b->doms[k].st->sp.size() + b->fns - 1) / b->fns; };
    auto tiles = [&](size_t k) {
        const Dims &d = b->doms[k].st->d;
        return ((d.nx + FCOLS - 1) / FCOLS) * ((d.ny + FROWS - 1) / FROWS);
    };
    auto columns = [&] {
        long long n = 0;
        for (size_t k = 0; k < b->doms.size(); k++) n += (long long)tiles(k) * groups(k);
        return n;
    };
    b->fns = 4;
    if (columns() < FILL / 2) b->fns = 2;
    const long long chunks = (FILL + columns() - 1) / columns();
    unsigned f = 0;
    for (size_t k = 0; k < b->doms.size(); k++) {
        const Dims &d = b->doms[k].st->d;
        const int S = (int)b->doms[k].st->sp.size(), ng = groups(k);
        const int kch = chunks >= d.nz ? 1 : (int)((d.nz + chunks - 1) / chunks);
        const int nk = (d.nz + kch - 1) / kch;
        for (int par = 0; par < 2; par++) {
            DomDesc &E = b->h_desc[par][k];
            E.f0 = f;
            E.ftx = (d.nx + FCOLS - 1) / FCOLS;
            E.fnk = nk;
            E.fkch = kch;
            E.fng = ng;
            E.fsb = S / ng;
            E.fsr = S % ng;
        }
        f += (unsigned)(tiles(k) * nk * ng);
    }
    b->total_fb = f;
}

std::string tune_key(const FastBatch *b)
{
    // batches of different storage classes run different kernel instantiations
    std::string k = std::to_string(b->order) + "/" + std::to_string(b->fct) + "/" +
                    std::to_string(storage_class(b));
    for (const auto &dm : b->doms)
        k += ":" + std::to_string(dm.st->d.nx) + "x" + std::to_string(dm.st->d.ny) + "x" +
             std::to_string(dm.st->d.nz) + "s" + std::to_string(dm.st->sp.size());
    return k;
}

}  // namespace

void launch_courant_b(const FastBatch *b, hipStream_t s, const DomDesc *D, int n)
{
    hipLaunchKernelGGL(k_courant_b, dim3(b->total_cb), dim3(64, 4), 0, s, D, n);
}

void launch_coef(const FastBatch *b, hipStream_t s, const DomDesc *D, int n)
{
    hipLaunchKernelGGL(k_coef, dim3(b->total_cb), dim3(64, 4), 0, s, D, n);
}

void launch_first(const FastBatch *b, hipStream_t s, const DomDesc *D, int n)
{
    const int fast = fast_division();
    auto go = [&](auto qk) {
        if (b->fns == 4)
            hipLaunchKernelGGL((k_first<qk.value, 4>), dim3(b->total_fb), dim3(64 * FWAVES), 0, s, D, n, fast);
        else
            hipLaunchKernelGGL((k_first<qk.value, 2>), dim3(b->total_fb), dim3(64 * FWAVES), 0, s, D, n, fast);
    };
    switch (storage_class(b)) {
    case QK_F32: go(std::integral_constant<int, QK_F32>{}); break;
    case QK_BF16: go(std::integral_constant<int, QK_BF16>{}); break;
    default: go(std::integral_constant<int, QK_ANY>{}); break;
    }
}

int fast_batch_tune(FastBatch *b, hipStream_t s, std::string *err)
{
    if (b->tuned) return 0;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
        return 0;  // never time inside a graph capture: keep the defaults
    const bool fix_cfg = getenv("ICAR_ADV_CORR_CFG") != nullptr;
    const bool fix_ks = getenv("ICAR_ADV_KSPLIT") != nullptr;
    const bool cached = !fix_cfg && !fix_ks;  // results with a fixed part are not shared
    const std::string key = tune_key(b);
    if (cached) {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        auto it = g_tuned.find(key);
        if (it != g_tuned.end()) {
            b->corr_cfg = it->second.first;
            b->tj = tile_rows(b->corr_cfg);
            set_ksplit(b, it->second.second);
            b->tuned = true;
            return 0;
        }
    }
    // candidates: the tiles, and column chunks while one chunk per column
    // leaves the GPU with few blocks
    std::vector<int> cfgs = fix_cfg ? std::vector<int>{b->corr_cfg}
                                    : std::vector<int>{3, 7, 6};
    const int n = (int)b->doms.size();
    const int par = b->doms[0].st->cur;
    // The timed launches are pass 2, which writes only the FP32 pass buffer
    // (order >= 3) or the alternate home buffer (order 2): both are written
    // again by the step that follows before anything reads them.  Its inputs
    // are made first, as the step makes them (Courant numbers, coefficients
    // and the donor-cell pass of the current state): timed on the real data,
    // the candidates take the path the step will take.
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return 0;
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return 0;
    }
    int rc = 0;
    if (b->dirty && (rc = upload_tables(b, s, err))) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        return rc;
    }
    {
        const DomDesc *D0 = b->d_desc + (size_t)par * n;
        launch_courant_b(b, s, D0, n);
        launch_coef(b, s, D0, n);
        launch_first(b, s, D0, n);
    }
    float best = 1e30f;
    int best_cfg = b->corr_cfg, best_ks = b->nks;
    for (int tj : {16, 8}) {
      std::vector<int> tcfgs;
      for (int cfg : cfgs)
          if (tile_rows(cfg) == tj) tcfgs.push_back(cfg);
      if (tcfgs.empty()) continue;
      b->tj = tj;
      std::vector<int> kss{b->nks};
      if (!fix_ks) {
          set_ksplit(b, 1);
          const unsigned base = b->total_work;
          kss = {1};
          if (base < 4096)
              for (int k : {2, 3, 4, 6, 8})
                  if ((unsigned)k * base <= 16384) kss.push_back(k);
      }
      std::vector<std::vector<int>> seen;  // chunk counts already timed
      for (int ks : kss) {
        set_ksplit(b, ks);
        std::vector<int> sig;
        for (int k = 0; k < n; k++) sig.push_back(b->h_desc[0][k].nks);
        bool dup = false;
        for (const auto &v : seen) dup = dup || v == sig;
        if (dup) continue;
        seen.push_back(sig);
        if ((rc = upload_tables(b, s, err))) break;
        const DomDesc *D = b->d_desc + (size_t)par * n;
        for (int cfg : tcfgs) {
            launch_corr(b, s, D, n, 2, cfg);  // warm-up
            (void)hipEventRecord(e0, s);
            for (int r = 0; r < 2; r++) launch_corr(b, s, D, n, 2, cfg);
            (void)hipEventRecord(e1, s);
            if (hipEventSynchronize(e1) != hipSuccess) {
                *err = "autotuning launch failed";
                rc = ICAR_ADV_EINVAL;
                break;
            }
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            if (ms < best * 0.97f) {  // prefer the earlier (simpler) candidate on near-ties
                best = ms;
                best_cfg = cfg;
                best_ks = ks;
            }
        }
        if (rc) break;
      }
      if (rc) break;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    b->corr_cfg = best_cfg;
    b->tj = tile_rows(best_cfg);
    set_ksplit(b, best_ks);
    b->tuned = true;
    if (cached) {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tuned[key] = {best_cfg, best_ks};
    }
    return 0;
}

void fast_batch_config(const FastBatch *b, int *corr_cfg, int *ksplit)
{
    if (corr_cfg) *corr_cfg = b ? b->corr_cfg : -1;
    if (ksplit) *ksplit = b ? b->h_desc[0][0].nks : -1;
}

FastBatch *fast_batch_create(const FastDomain *doms, int n, int order, int fct, std::string *err,
                             int *code)
{
    *code = ICAR_ADV_EINVAL;
    if (n < 1 || order < 1 || order > MAXP) {
        *err = "a batch needs at least one domain and 1 <= mpdata_order <= 16";
        return nullptr;
    }
    FastBatch *b = new FastBatch();
    b->doms.assign(doms, doms + n);
    b->order = order;
    b->fct = fct;
    // launch configuration: ICAR_ADV_CORR_CFG (0..7) and ICAR_ADV_KSPLIT fix
    // it, ICAR_ADV_AUTOTUNE=0 keeps the defaults; otherwise the first step
    // times the candidates on this batch
    const char *ec = getenv("ICAR_ADV_CORR_CFG"), *ek = getenv("ICAR_ADV_KSPLIT");
    const char *ea = getenv("ICAR_ADV_AUTOTUNE");
    if (ec) b->corr_cfg = atoi(ec) & 7;
    b->tj = tile_rows(b->corr_cfg);
    if (ek) b->nks = atoi(ek) < 1 ? 1 : atoi(ek);
    b->tuned = (ec && ek) || (ea && atoi(ea) == 0) || order < 2;
    unsigned cb = 0;
    for (int i = 0; i < 2; i++) b->h_desc[i].resize(n);
    for (int k = 0; k < n; k++) {
        FastState *st = doms[k].st;
        if (st->N >= 4294967296ull) {
            *err = "the fused path needs nx*ny*nz < 2^32 per domain";
            delete b;
            return nullptr;
        }
        if (st->sp.empty()) {
            *err = "a domain of the batch has no species bound";
            delete b;
            return nullptr;
        }
        // (a failed allocation leaves them out)
        if (std::count(st->alt.begin(), st->alt.end(), nullptr) > 0) {
            *code = ICAR_ADV_ENOMEM;
            *err = "a domain of the batch has a species without its second buffer";
            delete b;
            return nullptr;
        }
        if (st->tab_order != order && (*code = build_tables(st, order))) {
            *err = st->err;
            delete b;
            return nullptr;
        }
        *code = ICAR_ADV_EINVAL;
        b->gens.push_back(st->gen);
        const Dims &d = st->d;
        const int S = (int)st->sp.size();
        DomDesc D{};
        D.d = d;
        D.cb0 = cb;
        D.bx = (unsigned)((d.nx + 63) / 64);
        D.tiles_x = (d.nx + CTI - 1) / CTI;
        D.nspec = S;
        D.dx = doms[k].dx;
        D.dt = 0.0f;
        D.advect_density = doms[k].advect_density;
        D.compensated = doms[k].compensated;
        D.f = doms[k].f;
        D.sf = doms[k].sf;
        D.coef = st->coef;
        D.step = st->d_step;
        for (const FastSpecies &f : st->sp) {
            b->has_sr = b->has_sr || f.storage == ICAR_ADV_STORE_BF16_SR ||
                        f.storage == ICAR_ADV_STORE_F16_SR;
            b->q16 = b->q16 || f.storage != ICAR_ADV_STORE_F32;
            b->f16 = b->f16 || f.storage == ICAR_ADV_STORE_F16 || f.storage == ICAR_ADV_STORE_F16_SR;
        }
        cb += cell_blocks(d);
        b->cells += (double)st->N;
        b->cell_species += (double)st->N * S;
        for (int par = 0; par < 2; par++) {
            DomDesc E = D;
            for (int pass = 1; pass <= order; pass++)
                E.pass[pass - 1] = st->d_tab + ((size_t)par * order + (pass - 1)) * S;
            b->h_desc[par][k] = E;
        }
    }
    b->total_cb = cb;
    set_first_blocks(b);
    set_ksplit(b, b->nks);
    *code = ICAR_ADV_ENOMEM;
    if (hipMalloc(&b->d_desc, 2 * (size_t)n * sizeof(DomDesc)) != hipSuccess) {
        *err = "hipMalloc of the domain table failed";
        fast_batch_destroy(b);
        return nullptr;
    }
    // ring-condition table: every species of every domain, at both parities
    std::vector<BcEntry> bc[2];
    for (int k = 0; k < n; k++) {
        FastState *st = doms[k].st;
        const Dims &d = st->d;
        for (int s = 0; s < (int)st->sp.size(); s++)
            for (int par = 0; par < 2; par++)
                bc[par].push_back({d, home(st, s, par), (int)kind_bytes(st->sp[s].storage)});
    }
    b->n_bc = (int)bc[0].size();
    if (b->n_bc > 0) {
        const size_t nb = (size_t)b->n_bc * sizeof(BcEntry);
        if (hipMalloc(&b->d_bc, 2 * nb) != hipSuccess ||
            hipMemcpy(b->d_bc, bc[0].data(), nb, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(b->d_bc + b->n_bc, bc[1].data(), nb, hipMemcpyHostToDevice) != hipSuccess) {
            *err = "the ring-condition table could not be set up on the device";
            fast_batch_destroy(b);
            return nullptr;
        }
    }
    *code = 0;
    return b;
}

int fast_batch_bc(const FastBatch *b, hipStream_t s, int bc_x, int bc_y)
{
    if (b->n_bc == 0 || (bc_x == 0 && bc_y != 2)) return 0;
    const BcEntry *tab = b->d_bc + (size_t)b->doms[0].st->cur * b->n_bc;
    unsigned n = 0;
    for (const auto &dm : b->doms)
        n = std::max(n, ring_x_threads(dm.st->d, bc_x) + ring_y_threads(dm.st->d, bc_y));
    hipLaunchKernelGGL(k_bc_all, dim3(n / 256, b->n_bc), dim3(256), 0, s, tab, bc_x, bc_y);
    return (int)hipGetLastError();
}

void fast_batch_destroy(FastBatch *b)
{
    if (!b) return;
    (void)hipFree(b->d_desc);
    (void)hipFree(b->d_bc);
    delete b;
}

int fast_batch_prepare(FastBatch *b, hipStream_t s, const float *dt, std::string *err)
{
    const int n = (int)b->doms.size();
    for (int k = 0; k < n; k++)
        if (b->doms[k].st->gen != b->gens[k]) {
            *err = "species were re-bound after the batch was built";
            return ICAR_ADV_EINVAL;
        }
    bool same = (int)b->dts.size() == n;
    for (int k = 0; same && k < n; k++) same = b->dts[k] == dt[k];
    if (same && !b->dirty) return 0;
    b->dts.assign(dt, dt + n);
    for (int par = 0; par < 2; par++)
        for (int k = 0; k < n; k++) b->h_desc[par][k].dt = dt[k];
    if (b->dirty) return upload_tables(b, s, err);
    for (int d0 = 0; d0 < n; d0 += DT_SET) {
        DtSet v{};
        v.d0 = d0;
        v.n = std::min(n - d0, DT_SET);
        std::copy(dt + d0, dt + d0 + v.n, v.dt);
        hipLaunchKernelGGL(k_set_dt, dim3(1), dim3(DT_SET), 0, s, b->d_desc, n, v);
    }
    return 0;
}

int fast_batch_ready(FastBatch *b, hipStream_t s, const float *dt, std::string *err)
{
    int rc = fast_batch_prepare(b, s, dt, err);
    if (rc || b->tuned) return rc;
    if ((rc = fast_batch_tune(b, s, err))) return rc;
    return fast_batch_prepare(b, s, dt, err);
}

int fast_batch_advect(FastBatch *b, hipStream_t s, const float *dt, bool winds,
                      const TimedFn &timed, std::string *err)
{
    int rc = fast_batch_ready(b, s, dt, err);
    if (rc) return rc;
    const int n = (int)b->doms.size();
    const int par = b->doms[0].st->cur;
    for (int k = 1; k < n; k++)
        if (b->doms[k].st->cur != par) {
            *err = "the domains of the batch are at different buffer parities";
            return ICAR_ADV_EINVAL;
        }
    const DomDesc *D = b->d_desc + (size_t)par * n;
    const double cells = b->cells, cs = b->cell_species;
    if (winds) {
        // Courant numbers: reads u, v, w, density, jacobians, dz; writes 6 fields
        timed(K_COURANT, (9.0 + 6.0) * 4 * cells, [&] { launch_courant_b(b, s, D, n); });
        // species-invariant coefficients: reads U, V, Wd, G; writes NCOEF
        timed(K_COEF, (4.0 + NCOEF) * 4 * cells, [&] { launch_coef(b, s, D, n); });
    }
    // pass 1: donor cell for every species
    timed(K_FUSED_FIRST, 5.0 * 4 * cells + 2.0 * 4 * cs, [&] { launch_first(b, s, D, n); });
    for (int pass = 2; pass <= b->order; pass++) {
        // species read (q0 and q1 at pass 2) and written once; coefficients,
        // G, Gz and dz once
        const double bytes = (pass == 2 ? 3.0 : 2.0) * 4 * cs + (NCOEF + 3.0) * 4 * cells;
        timed(K_FUSED_CORR, bytes, [&] { launch_corr(b, s, D, n, pass, b->corr_cfg); });
    }
    if (b->has_sr)  // next step's rounding draws
        hipLaunchKernelGGL(k_tick, dim3((n + 63) / 64), dim3(64), 0, s, b->d_desc + (size_t)par * n, n);
    if (b->order <= 2)  // the results landed in the other home buffers
        for (auto &dm : b->doms) dm.st->cur = 1 - dm.st->cur;
    return 0;
}

// ---------------------------------------------------------------------------
// One species at a time (kernel_variant 0)
// ---------------------------------------------------------------------------
// The same kernels, a launch per pass and species, in place: the species keep
// their buffers and share two pass buffers, a and b.
//   order 1   q -> a (the caller copies a to q)
//   order 2   q -> a, with q copied to b; (b, a) -> q
//   order 3+  q -> a; (q, a) -> b; then b -> a, a -> b, ..., -> q
struct PlainState {
    FastState fs;        // the domain with one species, for the launch sizes
    FastBatch b;
    int order = 0;
    float *coef = nullptr, *a = nullptr, *c = nullptr;
    unsigned *d_step = nullptr; // the tables' allocation: two flags, then
    DomDesc *d_desc = nullptr;  // one per species
    SpecPass *d_tab = nullptr;  // [species][pass]
    std::vector<float *> q;     // the species and fields the tables are for
    DomainFields f{};
};

PlainState *plain_create(Dims d, int order, int fct)
{
    // ICAR_ADV_PASS_KERNELS=0: the kernel per subroutine and its 7 work fields
    const char *env = getenv("ICAR_ADV_PASS_KERNELS");
    if (env && *env && atoi(env) == 0) return nullptr;
    PlainState *st = new PlainState();
    st->order = order;
    st->fs.d = d;
    st->fs.N = (size_t)d.nx * d.ny * d.nz;
    st->fs.sp.assign(1, {nullptr, ICAR_ADV_STORE_F32, 0});
    st->b.order = order;
    st->b.fct = fct;
    st->b.total_cb = cell_blocks(d);
    st->b.doms.resize(1);
    st->b.doms[0].st = &st->fs;
    for (auto &h : st->b.h_desc) h.resize(1);
    // the tile and the column chunks: 16-row tiles where they fill the GPU
    // several times over, else 8-row tiles in as many chunks as make about
    // four blocks per CU
    auto tiles = [&](int tj) { return ((d.nx + CTI - 1) / CTI) * ((d.ny + tj - 1) / tj); };
    st->b.corr_cfg = tiles(16) >= 4096 ? 3 : 6;
    st->b.tj = tile_rows(st->b.corr_cfg);
    set_ksplit(&st->b, st->b.corr_cfg == 3 ? 1 : (1024 + tiles(8) / 2) / tiles(8));
    set_first_blocks(&st->b);
    // the tables of as many species as there can be, so that no step allocates
    constexpr size_t NS = ICAR_ADV_MAX_SPECIES, FLAGS = 256;  // [0] unused, [1] set by plain_coef
    static_assert(NS * sizeof(DomDesc) % alignof(SpecPass) == 0, "the pass table follows");
    const size_t fb = st->fs.N * sizeof(float);
    char *tables = nullptr;
    if (hipMalloc(&st->a, fb) != hipSuccess ||
        (order > 1 && (hipMalloc(&st->c, fb) != hipSuccess || hipMalloc(&st->coef, NCOEF * fb) != hipSuccess)) ||
        hipMalloc(&tables, FLAGS + NS * (sizeof(DomDesc) + (size_t)order * sizeof(SpecPass))) != hipSuccess) {
        (void)hipGetLastError();  // the caller takes the kernels that need less memory
        plain_destroy(st);
        return nullptr;
    }
    st->d_step = (unsigned *)tables;
    st->d_desc = (DomDesc *)(tables + FLAGS);
    st->d_tab = (SpecPass *)(st->d_desc + NS);
    return st;
}

void plain_destroy(PlainState *st)
{
    if (!st) return;
    void *bufs[] = {st->coef, st->a, st->c, st->d_step};
    for (void *p : bufs) (void)hipFree(p);
    delete st;
}

float *plain_result(PlainState *st) { return st->a; }

int plain_prepare(PlainState *st, hipStream_t s, const std::vector<float *> &q, const DomainFields &f,
                  const StepFields &sf, std::string *err)
{
    const int n = (int)q.size(), P = st->order;
    if (n == 0 || (q == st->q && memcmp(&f, &st->f, sizeof(f)) == 0)) return 0;
    st->q.clear();
    if (hipStreamSynchronize(s) != hipSuccess) {
        *err = "a previous step failed";
        return ICAR_ADV_EINVAL;
    }
    if (n > ICAR_ADV_MAX_SPECIES) {
        *err = "more species than the pass tables hold";
        return ICAR_ADV_ERANGE;
    }
    DomDesc D = st->b.h_desc[0][0];  // the launch sizes
    D.d = st->fs.d;
    D.cb0 = 0;
    D.bx = (unsigned)((D.d.nx + 63) / 64);
    D.tiles_x = (D.d.nx + CTI - 1) / CTI;
    D.nspec = 1;
    D.f = f;
    D.sf = sf;
    D.coef = st->coef;
    D.step = st->d_step;
    D.keep = P == 2 ? st->c : nullptr;
    std::vector<DomDesc> hd(n, D);
    std::vector<SpecPass> ht((size_t)n * P);
    for (int k = 0; k < n; k++)
        for (int p = 1; p <= P; p++) {
            SpecPass e{};
            e.kind0 = e.kindo = ICAR_ADV_STORE_F32;
            e.scale0 = e.inv_scaleo = 1.0f;
            float *const pass_buf[2] = {st->c, st->a};  // results of even and odd passes
            if (p == 1) {
                e.q0 = q[k];
            } else if (p == 2) {
                e.q0 = P == 2 ? st->c : q[k];
                e.q1 = st->a;
            } else {
                e.q0 = pass_buf[(p - 1) & 1];
            }
            e.out = p == P && P > 1 ? q[k] : pass_buf[p & 1];
            ht[(size_t)k * P + p - 1] = e;
            hd[k].pass[p - 1] = st->d_tab + (size_t)k * P + p - 1;
        }
    if (hipMemcpy(st->d_tab, ht.data(), ht.size() * sizeof(SpecPass), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(st->d_desc, hd.data(), hd.size() * sizeof(DomDesc), hipMemcpyHostToDevice) != hipSuccess) {
        *err = "upload of the species pass tables failed";
        return ICAR_ADV_ENOMEM;
    }
    st->q = q;
    st->f = f;
    return 0;
}

namespace {
__global__ void k_clear(unsigned *flag) { *flag = 0u; }
}  // namespace

void plain_coef(PlainState *st, hipStream_t s)
{
    if (st->q.empty()) return;  // no species was prepared: no table to read
    hipLaunchKernelGGL(k_clear, dim3(1), dim3(1), 0, s, st->d_step + 1);
    launch_coef(&st->b, s, st->d_desc, 1);
}

void plain_pass(PlainState *st, hipStream_t s, int species, int pass)
{
    if (species < 0 || species >= (int)st->q.size()) return;  // no table entry
    if (pass == 1) launch_first(&st->b, s, st->d_desc + species, 1);
    else launch_corr(&st->b, s, st->d_desc + species, 1, pass, st->b.corr_cfg);
}

void launch_pack(hipStream_t s, size_t n, const float *src, void *dst, int storage, int pow2);
void launch_unpack(hipStream_t s, size_t n, const void *src, float *dst, int storage, int pow2);

namespace {

__global__ void k_pack(size_t n, const float *__restrict__ src, uint16_t *__restrict__ dst,
                       int storage, float inv_scale)
{
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
         p += (size_t)gridDim.x * blockDim.x)
        dst[p] = to16(src[p], storage == ICAR_ADV_STORE_BF16_SR ? ICAR_ADV_STORE_BF16
                              : storage == ICAR_ADV_STORE_F16_SR ? ICAR_ADV_STORE_F16 : storage,
                      inv_scale, 0u);  // uploads round to nearest even
}

__global__ void k_unpack(size_t n, const uint16_t *__restrict__ src, float *__restrict__ dst,
                         int storage, float scale)
{
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
         p += (size_t)gridDim.x * blockDim.x)
        dst[p] = cvq<QK_ANY>(ldq<QK_ANY>(src, p, 0u, storage), storage, scale);
}

}  // namespace

void launch_pack(hipStream_t s, size_t n, const float *src, void *dst, int storage, int pow2)
{
    hipLaunchKernelGGL(k_pack, dim3(grid_for(n)), dim3(256), 0, s, n, src,
                       static_cast<uint16_t *>(dst), storage, ldexpf(1.0f, -pow2));
}

void launch_unpack(hipStream_t s, size_t n, const void *src, float *dst, int storage, int pow2)
{
    hipLaunchKernelGGL(k_unpack, dim3(grid_for(n)), dim3(256), 0, s, n,
                       static_cast<const uint16_t *>(src), dst, storage, ldexpf(1.0f, pow2));
}

}  // namespace icaradv
