// Velocity and temperature gradient sweeps of the viscous stages.
#include "cnd_ctx.hpp"

namespace cnd {

namespace {

// u, v, w, T of the state q at every stored point into prim (four fields NT
// apart), the arithmetic of SrcPrim, for the segmented eta and zeta sweeps.
__global__ __launch_bounds__(kPts) void k_prims(const BlkDev *__restrict__ blks, const Tile *__restrict__ tiles,
                                               const double *__restrict__ q, double *__restrict__ prim, int64_t NT)
{
    const Tile t = tiles[blockIdx.x];
    const BlkDev &B = blks[t.b];
    const int64_t npt = int64_t(B.n[0]) * B.n[1] * B.n[2];
    const int64_t lp = int64_t(t.q0) + threadIdx.x;
    if (lp >= npt) return;
    const int64_t g = B.off + lp;
    SrcPrim src{q, NT};
    SrcPrim::Raw raw;
    src.load(g, t.b, raw);
    double f[4];
    src.finish(raw, t.b, f);
#pragma unroll
    for (int m = 0; m < 4; ++m) prim[m * NT + g] = f[m];
}

}  // namespace

// The primitives lie in the flux scratch: the fluxes of the previous stage are
// consumed, and those of this one follow the gradient sweeps.
int run_prims(cnd_ctx *c, const double *cur)
{
    if (prims_wanted(c))
        LAUNCH(c, k_prims, pts_grid(c), dim3(kPts), 0, c->st, c->dblk, c->dpt, cur, c->fl, c->NT);
    return check_launch(c);
}

int run_grad(cnd_ctx *c, int d, const double *cur, bool joint)
{
    const int K = CND_KIND_GRAD;
    if (d > 0 && c->precision == CND_MIXED) {   // FP32 gradients (segmented only)
        LAUNCH_SEG_EZ((k_seg_grad_prim<G, float>), c, seg_launches(c, K, d, 1, joint), 1, 4, c->fl, c->gradf, c->NT)
    } else if (d > 0 && seg_on(c, K, d)) {
        LAUNCH_SEG_EZ((k_seg_grad_prim<G, double>), c, seg_launches(c, K, d, 1, joint), 1, 4, c->fl, c->grad, c->NT)
    } else
        LAUNCH_SWEEP(k_fd_grad, 4, c, d, 1, 4 * kTile, c->dblk, c->dtab, c->dlu, c->dtiles[d], ntiles(c, d), d,
                     c->nmax[d], c->ys, cur, c->grad, c->NT);
    return check_launch(c);
}

int run_grad_flux(cnd_ctx *c, const double *cur)
{
    const SegLaunches sls = seg_launches(c, CND_KIND_GRAD, 0, 4);
    if (c->precision == CND_MIXED) {
        LAUNCH_SEG_XI((k_seg_grad_flux<G, float>), c, sls, 1, 1, c->dinst, cur, c->gradf, c->met, c->fl, c->NT)
    } else {
        LAUNCH_SEG_XI((k_seg_grad_flux<G, double>), c, sls, 1, 1, c->dinst, cur, c->grad, c->met, c->fl, c->NT)
    }
    return check_launch(c);
}

}  // namespace cnd
