// Sources, sinks, sweep-shape table and sweep kernel templates of libcnd.
// Each sweep kind's launches (and so its template instantiations) live in a
// translation unit of their own (cnd_run_*.hip), so they compile in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "cnd_dev.hpp"
#include "cnd_kernels.hpp"
#include "cnd_seg.hpp"
#include "cnd_sweep.hpp"

namespace cnd {

// ---- sources (values a sweep differentiates or filters) ---------------------
template <int NV>
struct SrcField {   // NV plain fields, vs apart
    const double *a;
    int64_t vs;
    struct Raw { double v[NV]; };
    __device__ double field(int64_t g, int v) const { return a[v * vs + g]; }
    __device__ void load(int64_t g, int, Raw &r) const
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) r.v[k] = a[k * vs + g];
    }
    __device__ void finish(const Raw &r, int, double (&v)[NV]) const
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] = r.v[k];
    }
};

// u, v, w, T of the state q.
__device__ __forceinline__ void prims_of(const double (&q)[5], double (&o)[4])
{
    const double ri = 1.0 / q[0];
    const double u = q[1] * ri, v = q[2] * ri, w = q[3] * ri;
    const double p = kGm1 * (q[4] - 0.5 * ((q[1] * u + q[2] * v) + q[3] * w));
    o[0] = u; o[1] = v; o[2] = w;
    o[3] = (kGam * p) * ri;
}

// u, v, w, T of a state, exactly as the reference's primitives step
// (src/mo_canard_driver.f90:267-274).
struct SrcPrim {
    const double *q;
    int64_t NT;
    struct Raw { double q[5]; };
    __device__ void load(int64_t g, int, Raw &r) const
    {
#pragma unroll
        for (int m = 0; m < 5; ++m) r.q[m] = q[m * NT + g];
    }
    __device__ void finish(const Raw &r, int, double (&o)[4]) const
    {
        prims_of(r.q, o);
    }
};

// The five flux components of direction d at one point
// (src/mo_physics.f90:319-382): the inviscid part from the state q1..q5 and
// the metric row m of d, then, with stresses t (txx, tyy, tzz, txy, tyz,
// tzx and the three heat-flux rows), the viscous part.
template <bool VIS>
__device__ __forceinline__ void dir_flux(double q1, double q2, double q3, double q4, double q5, double u, double v,
                                         double w, double p, const double (&m)[3], const double *umf,
                                         const double *t, double (&o)[5])
{
    const double m0 = m[0], m1 = m[1], m2 = m[2];
    const double s = (m0 * (u + umf[0]) + m1 * (v + umf[1])) + m2 * (w + umf[2]);
    o[0] = q1 * s;
    o[1] = q2 * s + m0 * p;
    o[2] = q3 * s + m1 * p;
    o[3] = q4 * s + m2 * p;
    o[4] = (q5 + p) * s - p * ((umf[0] * m0 + umf[1] * m1) + umf[2] * m2);
    if constexpr (VIS) {
        // stress rows x (txx, txy, tzx), y (txy, tyy, tyz), z (tzx, tyz, tzz)
        const double txx = t[0], tyy = t[1], tzz = t[2], txy = t[3], tyz = t[4], tzx = t[5];
        o[1] = o[1] - m0 * txx; o[1] = o[1] - m1 * txy; o[1] = o[1] - m2 * tzx;
        o[2] = o[2] - m0 * txy; o[2] = o[2] - m1 * tyy; o[2] = o[2] - m2 * tyz;
        o[3] = o[3] - m0 * tzx; o[3] = o[3] - m1 * tyz; o[3] = o[3] - m2 * tzz;
        o[4] = o[4] - m0 * t[6]; o[4] = o[4] - m1 * t[7]; o[4] = o[4] - m2 * t[8];
    }
}

// Sutherland's law in the reference's scaling (src/mo_physics.f90:245-247);
// T^1.5 as T sqrt(T): two roundings instead of a general power's ~200
// instructions.
__device__ __forceinline__ double viscosity(const InstDev &I, double T)
{
    return (I.srefp1dre * (T * sqrt(T))) / (T + I.srefoo);
}

// Viscous stresses and heat flux (src/mo_physics.f90:249-299) at point g and,
// from them, the fluxes of all three directions (src/mo_physics.f90:319-382)
// into F[5 d + m]: gx the xi gradients of u, v, w, T, grad the stored ones
// (fields 4 .. 11: eta and zeta).
template <class TG>
__device__ __forceinline__ void visc_point(const InstDev &I, int64_t g, const double (&gx)[4], const double *q,
                                           const TG *grad, const double *met, double *F, int64_t NT)
{
    const double q1 = q[g], q5 = q[4 * NT + g];
    const double q2 = q[NT + g], q3 = q[2 * NT + g], q4 = q[3 * NT + g];
    double ge[4], gz[4], mt[9];
#pragma unroll
    for (int k = 0; k < 4; ++k) ge[k] = double(grad[(4 + k) * NT + g]);
#pragma unroll
    for (int k = 0; k < 4; ++k) gz[k] = double(grad[(8 + k) * NT + g]);
#pragma unroll
    for (int c = 0; c < 9; ++c) mt[c] = met[c * NT + g];
    const double J = met[9 * NT + g];
    const double ri = 1.0 / q1;
    const double u = q2 * ri, v = q3 * ri, w = q4 * ri;
    const double p = kGm1 * (q5 - 0.5 * ((q2 * u + q3 * v) + q4 * w));
    const double T = (kGam * p) * ri;
    const double mu = viscosity(I, T);
    auto CT = [&](int c, int var) { return (mt[c] * gx[var] + mt[3 + c] * ge[var]) + mt[6 + c] * gz[var]; };
    const double vtxx = CT(0, 0), vhzz = CT(1, 0), vtzx = CT(2, 0);
    const double vtxy = CT(0, 1), vtyy = CT(1, 1), vhxx = CT(2, 1);
    const double vhyy = CT(0, 2), vtyz = CT(1, 2), vtzz = CT(2, 2);
    const double s1 = CT(0, 3), s2 = CT(1, 3), s3 = CT(2, 3);
    const double r1 = mu * J;
    const double r2 = kGm1PrI * r1;
    const double d5 = kTwoThirds * ((vtxx + vtyy) + vtzz);
    double ts[9];
    const double txx = r1 * ((vtxx + vtxx) - d5), tyy = r1 * ((vtyy + vtyy) - d5), tzz = r1 * ((vtzz + vtzz) - d5);
    const double txy = r1 * (vtxy + vhzz), tyz = r1 * (vtyz + vhxx), tzx = r1 * (vtzx + vhyy);
    ts[0] = txx; ts[1] = tyy; ts[2] = tzz; ts[3] = txy; ts[4] = tyz; ts[5] = tzx;
    ts[6] = ((r2 * s1 + u * txx) + v * txy) + w * tzx;
    ts[7] = ((r2 * s2 + u * txy) + v * tyy) + w * tyz;
    ts[8] = ((r2 * s3 + u * tzx) + v * tyz) + w * tzz;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double m[3] = {mt[3 * d], mt[3 * d + 1], mt[3 * d + 2]};
        double o[5];
        dir_flux<true>(q1, q2, q3, q4, q5, u, v, w, p, m, I.umf, ts, o);
#pragma unroll
        for (int c = 0; c < 5; ++c) F[(5 * d + c) * NT + g] = o[c];
    }
}

// Inviscid fluxes (src/mo_physics.f90:319-382) of the state q1..q5 at point g
// into F[5 d + m]: of all three directions, or (not ALL) of those whose bit is
// set in dirs.
template <bool ALL>
__device__ __forceinline__ void inv_point(const InstDev &I, int64_t g, const double (&q)[5], const double *met,
                                          double *F, int64_t NT, unsigned dirs)
{
    const double ri = 1.0 / q[0];
    const double u = q[1] * ri, v = q[2] * ri, w = q[3] * ri;
    const double p = kGm1 * (q[4] - 0.5 * ((q[1] * u + q[2] * v) + q[3] * w));
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!ALL && !(dirs >> d & 1)) continue;
        const double m[3] = {met[(3 * d) * NT + g], met[(3 * d + 1) * NT + g], met[(3 * d + 2) * NT + g]};
        double o[5];
        dir_flux<false>(q[0], q[1], q[2], q[3], q[4], u, v, w, p, m, I.umf, nullptr, o);
#pragma unroll
        for (int c = 0; c < 5; ++c) F[(5 * d + c) * NT + g] = o[c];
    }
}

// Inviscid fluxes of direction d evaluated in a tiled sweep from q and the
// metric row of d, with inv_point's arithmetic.
struct SrcFlux {
    const double *q;
    const double *met;
    const BlkDev *blks;
    const InstDev *inst;
    int64_t NT;
    int d;
    struct Raw { double q[5], m[3]; };
    __device__ void load(int64_t g, int, Raw &r) const
    {
#pragma unroll
        for (int k = 0; k < 5; ++k) r.q[k] = q[k * NT + g];
#pragma unroll
        for (int k = 0; k < 3; ++k) r.m[k] = met[(3 * d + k) * NT + g];
    }
    __device__ void finish(const Raw &r, int b, double (&o)[5]) const
    {
        const double q1 = r.q[0], q2 = r.q[1], q3 = r.q[2], q4 = r.q[3], q5 = r.q[4];
        const double ri = 1.0 / q1;
        const double u = q2 * ri, v = q3 * ri, w = q4 * ri;
        const double p = kGm1 * (q5 - 0.5 * ((q2 * u + q3 * v) + q4 * w));
        dir_flux<false>(q1, q2, q3, q4, q5, u, v, w, p, r.m, inst[blks[b].inst].umf, nullptr, o);
    }
};

// ---- sinks ----------------------------------------------------------------
// store writes results; fold(f, x) is the value to write for source f
// and result x, written with put_raw by sweeps that still hold the source in
// registers (the filter adds its correction to the source).
template <int NV, class TO = double>
struct SinkOut {   // out fields vs apart, stored as TO
    TO *o;
    int64_t vs;
    __device__ void store(int64_t g, int, const double (&x)[NV])
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) o[k * vs + g] = TO(x[k]);
    }
    static constexpr bool kReadBack = false;
    __device__ double fold(double, double x) const { return x; }
    __device__ void put_raw(int64_t g, int, int k, double x) { o[k * vs + g] = TO(x); }
    __device__ void ends(int, int, int, double) {}
};

// The xi gradients of u, v, w, T straight into the point's stresses and fluxes.
template <class TG>
struct SinkVisc {
    const InstDev *I;
    const double *q;
    const TG *grad;
    const double *met;
    double *F;
    int64_t NT;
    __device__ void store(int64_t g, int, const double (&x)[4]) { visc_point(*I, g, x, q, grad, met, F, NT); }
    static constexpr bool kReadBack = false;
    __device__ void ends(int, int, int, double) {}
};

template <int NV>
struct SinkFilt {  // out = f + correction
    double *o;
    const double *f;
    int64_t vs;
    __device__ void store(int64_t g, int, const double (&x)[NV])
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) o[k * vs + g] = f[k * vs + g] + x[k];
    }
    static constexpr bool kReadBack = true;   // results are added to the sources
    __device__ double src(int64_t g, int k) const { return f[k * vs + g]; }
    __device__ double fold(double fv, double x) const { return fv + x; }
    __device__ void put_raw(int64_t g, int, int k, double x) { o[k * vs + g] = x; }
    __device__ void ends(int, int, int, double) {}
};

struct SinkFlux {  // the five components of dF/dxi_d; pencil ends to drva
    double *de, *drva;
    int64_t NT, FT, fi0;
    __device__ void store(int64_t g, int, const double (&x)[5])
    {
#pragma unroll
        for (int m = 0; m < 5; ++m) de[m * NT + g] = x[m];
    }
    __device__ void ends(int side, int lane, int m, double x) { drva[(side * 5 + m) * FT + fi0 + lane] = x; }
};

struct SinkFluxV {  // component v of dF/dxi_d; pencil ends to drva
    double *o, *drva;
    int v;
    int64_t FT, fi0;
    __device__ void store(int64_t g, int, const double (&x)[1]) { o[g] = x[0]; }
    static constexpr bool kReadBack = false;
    __device__ double fold(double, double x) const { return x; }
    __device__ void put_raw(int64_t g, int, int, double x) { o[g] = x; }
    __device__ void ends(int side, int lane, int, double x) { drva[(side * 5 + v) * FT + fi0 + lane] = x; }
};

// Component v of the last flux derivative folded straight into the RK update
// (k_update's arithmetic without the sponge, same operation order, so results
// are bit-identical): qa = qo - dt/(5-nk) * yaco * ((de_xi + de_eta) + de_zeta),
// where the sweep's own result x is de_zeta (XFIRST false: da, db the xi and
// eta buffers) or de_xi (XFIRST true: da, db the eta and zeta buffers).
// Every operand is variable v at the sink's own point.  Pre holds one point's
// operands, so sweeps can load them for several points before storing any.
template <bool XFIRST>
struct SinkUpdateV {
    double *qa, *drva;
    const double *qo, *da, *db, *met;
    double dtk;   // dt / (5 - nk) of the tile's instance
    int v;
    int64_t NT, FT, fi0;
    struct Pre { double a, b, q, r; };
    __device__ void pre(int64_t g, Pre &o) const
    {
        o.a = da[g];
        o.b = db[g];
        o.q = qo[g];
        o.r = dtk * met[9 * NT + g];
    }
    __device__ void put_pre(int64_t g, double x, const Pre &o)
    {
        const double s = XFIRST ? (x + o.a) + o.b : (o.a + o.b) + x;
        qa[g] = o.q - o.r * s;
    }
    static constexpr bool kReadBack = false;
    __device__ void ends(int side, int lane, int, double x) { drva[(side * 5 + v) * FT + fi0 + lane] = x; }
};

// ---- sweep kernels -----------------------------------------------------------
// grid: (xcd_width(tiles of direction d), variable groups); NV waves per tile
// of 64 pencils; C = chunk_of(d); dynamic LDS = sweep_lds_bytes<NV, C>().
#define SWEEP_TILE_PROLOGUE(ntiles)        \
    const int tix = xcd_tile(ntiles);      \
    if (tix >= (ntiles)) return;           \
    extern __shared__ double lds[];

template <int C>
__global__ __launch_bounds__(kTile) void k_fd_field(const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs,
                                                   const double *__restrict__ lu, const Tile *__restrict__ tiles,
                                                   int ntiles, int d, int n45, int nmax, double *ys,
                                                   const double *in, int64_t in_vstride, double *out,
                                                   int64_t out_vstride)
{
    SWEEP_TILE_PROLOGUE(ntiles)
    const int v = blockIdx.y;
    SrcField<1> src{in + v * in_vstride, 0};
    SinkOut<1> sink{out + v * out_vstride, 0};
    sweep_tile<1, 0, C>(blks, tabs, lu, tiles[tix], int64_t(v) * ntiles + tix, d, n45, nmax, ys, src, sink, lds);
}

template <int C>
__global__ __launch_bounds__(kTile) void k_filter_field(const BlkDev *__restrict__ blks,
                                                       const TabDev *__restrict__ tabs,
                                                       const double *__restrict__ lu,
                                                       const Tile *__restrict__ tiles, int ntiles, int d, int nmax,
                                                       double *ys, const double *in, double *out, int64_t vstride)
{
    SWEEP_TILE_PROLOGUE(ntiles)
    const int v = blockIdx.y;
    SrcField<1> src{in + v * vstride, 0};
    SinkFilt<1> sink{out + v * vstride, in + v * vstride, 0};
    sweep_tile<1, 1, C>(blks, tabs, lu, tiles[tix], int64_t(v) * ntiles + tix, d, 0, nmax, ys, src, sink, lds);
}

// Velocity and temperature gradients along d (the 12 derivative sweeps of
// calc_viscous_shear_stress, src/mo_physics.f90:238-280).
template <int C>
__global__ __launch_bounds__(4 * kTile) void k_fd_grad(const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs,
                                                  const double *__restrict__ lu, const Tile *__restrict__ tiles,
                                                  int ntiles, int d, int nmax, double *ys, const double *q,
                                                  double *grad, int64_t NT)
{
    SWEEP_TILE_PROLOGUE(ntiles)
    SrcPrim src{q, NT};
    SinkOut<4> sink{grad + 4 * d * NT, NT};
    sweep_tile<4, 0, C>(blks, tabs, lu, tiles[tix], tix, d, 0, nmax, ys, src, sink, lds);
}

// Flux derivatives along d (src/mo_physics.f90:385-399) into the d-th
// right-hand-side buffer de: inviscid fluxes evaluated in the sweep, five
// waves on one tile.  With stored fluxes in a sweep per component, as the
// segmented sweeps take them, a step of 601 x 561 x 541 points went from 154
// to 177 ms: the forward values' scratch makes these sweeps bound by their
// bytes, and the stored fluxes add 20 fields a stage to them.
template <int C>
__global__ __launch_bounds__(5 * kTile) void k_fd_flux(const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs,
                                                  const InstDev *__restrict__ inst, const double *__restrict__ lu,
                                                  const Tile *__restrict__ tiles, int ntiles, int d, int nmax,
                                                  double *ys, const double *q, const double *met, double *de,
                                                  double *drva, int64_t NT, int64_t FT)
{
    SWEEP_TILE_PROLOGUE(ntiles)
    const Tile t = tiles[tix];
    SrcFlux src{q, met, blks, inst, NT, d};
    SinkFlux sink{de, drva, NT, FT, blks[t.b].foff[d] + t.q0};
    sweep_tile<5, 0, C>(blks, tabs, lu, t, tix, d, 0, nmax, ys, src, sink, lds);
}

// ... or stored fluxes F (component v = blockIdx.y), the viscous case.
template <int C>
__global__ __launch_bounds__(kTile) void k_fd_flux_field(const BlkDev *__restrict__ blks,
                                                        const TabDev *__restrict__ tabs,
                                                        const double *__restrict__ lu, const Tile *__restrict__ tiles,
                                                        int ntiles, int d, int nmax, double *ys, const double *F,
                                                        double *de, double *drva, int64_t NT, int64_t FT)
{
    SWEEP_TILE_PROLOGUE(ntiles)
    const int v = blockIdx.y;
    const Tile t = tiles[tix];
    SrcField<1> src{F + v * NT, 0};
    SinkFluxV sink{de + v * NT, drva, v, FT, blks[t.b].foff[d] + t.q0};
    sweep_tile<1, 0, C>(blks, tabs, lu, t, int64_t(v) * ntiles + tix, d, 0, nmax, ys, src, sink, lds);
}

// ---- segmented sweeps (cnd_seg.hpp) ---------------------------------------
// Compiled shapes: L points per segment (lanes per pencil = segments =
// ceil(n / L)), P pencils per workgroup, at most SPMAX segments per pencil; XI
// shapes stage runs along the pencil (xi sweeps), the others take P
// neighbouring pencils (eta, zeta sweeps).  C is the run length reported with
// a shape; no sweep stages in runs of it any more, so shapes that differ in C
// only are the same.  The autotuner picks one per sweep kind and direction.
// Short segments suit small blocks, where a sweep is one wave's chain of
// instructions (17 -> 9 points: eta and zeta filters 9.7 -> 7.3 us at 17^3,
// 10.2 -> 8.2 us at 33^3, 14.2 -> 12.0 us at 101 x 61 x 41); long ones run
// fewer scans and closure rows per point (257^3: 33 points).
template <int L_, int P_, int C_, int SPMAX_, bool XI_>
struct SegG { static constexpr int L = L_, P = P_, C = C_, SPMAX = SPMAX_; static constexpr bool XI = XI_; };
struct ShapeInfo { int L, P, C, SPMAX; bool XI; };
constexpr int kNumShapes = 29;
constexpr ShapeInfo kShapes[kNumShapes] = {
    {17, 4, 16, 16, true},    // 0: xi default (pencils up to 272 points)
    {33, 4, 16, 8, true},     // 1
    {33, 16, 8, 8, false},    // 2: eta/zeta default (up to 264 points)
    {33, 16, 4, 8, false},    // 3
    {17, 8, 8, 16, false},    // 4
    {33, 4, 16, 16, true},    // 5: long xi pencils (up to 528 points)
    {33, 8, 8, 16, false},    // 6: long eta/zeta pencils (up to 528 points)
    {17, 8, 16, 16, true},    // 7: xi, wider tiles (single-field sweeps)
    {17, 16, 16, 16, true},   // 8
    {17, 16, 8, 16, false},   // 9: eta/zeta, short segments, wide tiles
    {33, 32, 8, 8, false},    // 10: eta/zeta, runs of 32 and 64 points
    {33, 64, 8, 8, false},    // 11
    {17, 32, 8, 16, false},   // 12
    {17, 64, 8, 16, false},   // 13
    {17, 32, 16, 16, true},   // 14: xi, 32-pencil tiles (single-field sweeps)
    {17, 20, 16, 16, true},   // 15: xi, tiles sized for three workgroups per CU
    {17, 24, 16, 16, true},   // 16
    // 17-point segments on pencils of up to 528 points: with 33-point ones a
    // workgroup has 4 pencils and half the waves (513-point xi pencils of
    // the four sheared blocks: flux 1.26 -> 0.89 ms beside the eta sweep,
    // filter 1.28 -> 0.64, gradients 0.63 -> 0.59)
    {17, 16, 16, 32, true},   // 17
    {17, 8, 16, 32, true},    // 18
    {17, 4, 16, 32, true},    // 19
    {17, 16, 8, 32, false},   // 20
    {9, 4, 16, 16, true},     // 21
    {9, 8, 16, 16, true},     // 22
    {9, 16, 16, 16, true},    // 23
    {9, 32, 16, 16, true},    // 24
    {9, 8, 8, 16, false},     // 25
    {9, 16, 8, 16, false},    // 26
    {9, 32, 8, 16, false},    // 27
    {9, 64, 8, 16, false}};   // 28
using Sh0 = SegG<17, 4, 16, 16, true>;
using Sh1 = SegG<33, 4, 16, 8, true>;
using Sh2 = SegG<33, 16, 8, 8, false>;
using Sh3 = Sh2;   // differs in the reported run length only
using Sh4 = SegG<17, 8, 8, 16, false>;
using Sh5 = SegG<33, 4, 16, 16, true>;
using Sh6 = SegG<33, 8, 8, 16, false>;
using Sh7 = SegG<17, 8, 16, 16, true>;
using Sh8 = SegG<17, 16, 16, 16, true>;
using Sh9 = SegG<17, 16, 8, 16, false>;
using Sh10 = SegG<33, 32, 8, 8, false>;
using Sh11 = SegG<33, 64, 8, 8, false>;
using Sh12 = SegG<17, 32, 8, 16, false>;
using Sh13 = SegG<17, 64, 8, 16, false>;
using Sh14 = SegG<17, 32, 16, 16, true>;
using Sh15 = SegG<17, 20, 16, 16, true>;
using Sh16 = SegG<17, 24, 16, 16, true>;
using Sh17 = SegG<17, 16, 16, 32, true>;
using Sh18 = SegG<17, 8, 16, 32, true>;
using Sh19 = SegG<17, 4, 16, 32, true>;
using Sh20 = SegG<17, 16, 8, 32, false>;
using Sh21 = SegG<9, 4, 16, 16, true>;
using Sh22 = SegG<9, 8, 16, 16, true>;
using Sh23 = SegG<9, 16, 16, 16, true>;
using Sh24 = SegG<9, 32, 16, 16, true>;
using Sh25 = SegG<9, 8, 8, 16, false>;
using Sh26 = SegG<9, 16, 8, 16, false>;
using Sh27 = SegG<9, 32, 8, 16, false>;
using Sh28 = SegG<9, 64, 8, 16, false>;
// workgroup size bound of a kernel (shapes whose NV * P * SPMAX exceeds the
// 1024-thread limit are rejected at launch time by shape_sp)
__host__ __device__ constexpr int wg_bound(int x) { return x > 1024 ? 1024 : x; }
// waves per SIMD a segmented sweep is compiled for: eta / zeta sweeps of
// 17-point segments are held to 96 VGPRs (5 waves) where that costs no spills,
// not in the filter and the fused update, whose operands need more; other shapes of
// up to 17 points to 128 (4 waves; those of 9 points need 84 to 102 anyway,
// and forcing 80 spills), the others are left to the compiler.  4 -> 5 waves,
// 129^3: joint gradient sweeps 59 -> 53 us, flux sweeps 87 -> 86 us.
template <class G, bool OPERANDS = false>
__host__ __device__ constexpr int seg_waves() { return G::L > 17 ? 1 : (G::L == 17 && !G::XI && !OPERANDS ? 5 : 4); }
constexpr int kSegMaxPoints = 528;   // longest pencil of a segmented sweep
constexpr int kTiled = -1;   // shape index of the tiled sweep
// pencils-per-workgroup values (tile lists)
constexpr int kNumP = 7, kPs[kNumP] = {4, 8, 16, 32, 64, 20, 24};
__host__ __device__ constexpr int p_index(int P)
{
    return P == 4 ? 0 : (P == 8 ? 1 : (P == 16 ? 2 : (P == 32 ? 3 : (P == 64 ? 4 : (P == 20 ? 5 : 6)))));
}

// Tiles of one direction d (split = ntiles), or of eta and zeta in one launch
// (d = 1; tiles from split on are zeta's).
// list null: the tiles of a context of one block, whose place follows from
// their number (a dependent load less at the start of every workgroup).
struct SegTiles {
    const Tile *list;
    int n, SP, d, split;
    __device__ int dir(int tix) const { return d + (tix >= split ? 1 : 0); }
    __device__ Tile at(int tix, int P) const
    {
        return list ? list[tix] : Tile{0, (tix - (tix >= split ? split : 0)) * P};
    }
};
#define SEG_PROLOGUE                       \
    const int tix = xcd_tile(tiles.n);     \
    if (tix >= tiles.n) return;            \
    const int d = tiles.dir(tix);          \
    extern __shared__ double lds[];

template <class G>
__global__ __launch_bounds__(wg_bound(G::P * G::SPMAX), (seg_waves<G>())) void k_seg_fd_field(
    const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs, SegTabs tb, const SegTiles tiles, int n45,
    const double *in, int64_t in_vstride, double *out, int64_t out_vstride)
{
    SEG_PROLOGUE
    const int v = blockIdx.y;
    SrcField<1> src{in + v * in_vstride, 0};
    SinkOut<1> sink{out + v * out_vstride, 0};
    seg_tile<1, 0, G::L, G::P, G::XI>(blks, tabs, tb, tiles.at(tix, G::P), d, n45, tiles.SP, src, sink, lds);
}

template <class G>
__global__ __launch_bounds__(wg_bound(G::P * G::SPMAX), (seg_waves<G, true>())) void k_seg_filter_field(
    const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs, SegTabs tb, const SegTiles tiles,
    const double *in, double *out, int64_t vstride)
{
    SEG_PROLOGUE
    const int v = blockIdx.y;
    SrcField<1> src{in + v * vstride, 0};
    SinkFilt<1> sink{out + v * vstride, in + v * vstride, 0};
    seg_tile<1, 1, G::L, G::P, G::XI>(blks, tabs, tb, tiles.at(tix, G::P), d, 0, tiles.SP, src, sink, lds);
}

// Xi gradients of u, v, w, T and, from them and the stored eta and zeta ones
// (TG: float in mixed precision), the stresses and the fluxes of all three
// directions: a tile is one contiguous run of points, so the sink streams the
// point's other operands like a pointwise kernel.  The xi gradients are never
// stored: 344 B per point (40 of them the state again, mostly from the
// last-level cache) against 72 + 336 for a sweep and a pointwise kernel.
// 257^3, a stage: 0.386 + 1.087 -> 1.222 ms, and 0.221 for the primitives the
// separate sweep stored; 65^3: 16.3 + 15.3 -> 26.1 us.
template <class G, class TG>
__global__ __launch_bounds__(wg_bound(4 * G::P * G::SPMAX), (seg_waves<G>())) void k_seg_grad_flux(
    const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs, SegTabs tb, const SegTiles tiles,
    const InstDev *__restrict__ inst, const double *q, const TG *grad, const double *met, double *F, int64_t NT)
{
    SEG_PROLOGUE
    const Tile t = tiles.at(tix, G::P);
    SrcPrim src{q, NT};
    SinkVisc<TG> sink{inst + blks[t.b].inst, q, grad, met, F, NT};
    seg_tile<4, 0, G::L, G::P, G::XI>(blks, tabs, tb, t, d, 0, tiles.SP, src, sink, lds);
}

// Gradients along d (eta, zeta) of the primitive v = blockIdx.y (prim, four
// fields NT apart), into grad as TG.
template <class G, class TG>
__global__ __launch_bounds__(wg_bound(G::P * G::SPMAX), (seg_waves<G>())) void k_seg_grad_prim(
    const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs, SegTabs tb, const SegTiles tiles, const double *prim, TG *grad,
    int64_t NT)
{
    SEG_PROLOGUE
    const int v = blockIdx.y;
    SrcField<1> src{prim + v * NT, 0};
    SinkOut<1, TG> sink{grad + (4 * d + v) * NT, 0};
    seg_tile<1, 0, G::L, G::P, G::XI>(blks, tabs, tb, tiles.at(tix, G::P), d, 0, tiles.SP, src, sink, lds);
}

// Pencil-end derivatives of the three directions, and their face strides.
struct Ends3 { double *drva[3]; int64_t FT[3]; };

// Derivatives along d of the stored fluxes (component v = blockIdx.y) into the
// d-th right-hand-side buffer of de.
template <class G>
__global__ __launch_bounds__(wg_bound(G::P * G::SPMAX), (seg_waves<G>())) void k_seg_flux_field(
    const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs, SegTabs tb, const SegTiles tiles,
    const double *F, double *de, const Ends3 ends, int64_t NT)
{
    SEG_PROLOGUE
    const int v = blockIdx.y;
    const Tile t = tiles.at(tix, G::P);
    SrcField<1> src{F + (5 * d + v) * NT, 0};
    SinkFluxV sink{de + (5 * d + v) * NT, ends.drva[d], v, ends.FT[d], blks[t.b].foff[d] + t.q0};
    seg_tile<1, 0, G::L, G::P, G::XI>(blks, tabs, tb, t, d, 0, tiles.SP, src, sink, lds);
}

// Last flux sweep of a stage fused with the RK update: sweep of the stored
// flux component v along d (xi or zeta), written as the updated state qa.
// Grid x: five workgroups (components) per tile.
template <class G>
__global__ __launch_bounds__(wg_bound(G::P * G::SPMAX), (seg_waves<G, true>())) void k_seg_flux_update(
    const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs, SegTabs tb, const SegTiles tiles,
    const InstDev *__restrict__ inst, const double *F, const double *de, const double *__restrict__ qo,
    const double *__restrict__ met, double *qa, const Ends3 ends, int64_t NT, int nk)
{
    // the five component workgroups of a tile follow each other on one XCD,
    // so the Jacobian they all read is fetched once into that XCD's L2
    const int w = xcd_tile(5 * tiles.n);
    if (w >= 5 * tiles.n) return;
    extern __shared__ double lds[];
    const int tix = w / 5, v = w % 5, d = tiles.d;
    const Tile t = tiles.at(tix, G::P);
    SrcField<1> src{F + (5 * d + v) * NT, 0};
    const double dtk = inst[blks[t.b].inst].dt / double(4 - nk + 1);
    // the two other directions' right-hand sides
    const double *da = de + ((G::XI ? 5 : 0) + v) * NT, *db = de + ((G::XI ? 10 : 5) + v) * NT;
    SinkUpdateV<G::XI> sink{qa + v * NT, ends.drva[d], qo + v * NT, da, db, met, dtk, v, NT, ends.FT[d],
                            blks[t.b].foff[d] + t.q0};
    seg_tile<1, 0, G::L, G::P, G::XI>(blks, tabs, tb, t, d, 0, tiles.SP, src, sink, lds);
}

}  // namespace cnd
