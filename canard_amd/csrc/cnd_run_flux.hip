// Flux derivative sweeps into the right-hand-side buffers.
#include "cnd_ctx.hpp"

namespace cnd {

int run_flux(cnd_ctx *c, int d, const double *cur, bool joint)
{
    const int K = CND_KIND_FLUX;
    if (seg_on(c, K, d))
        LAUNCH_SEG((k_seg_flux_field<G>), c, seg_launches(c, K, d, 1, joint), 1, 5, c->fl, c->de, ends3(c), c->NT);
    else if (!c->any_visc)
        LAUNCH_SWEEP(k_fd_flux, 5, c, d, 1, 5 * kTile, c->dblk, c->dtab, c->dinst, c->dlu, c->dtiles[d], ntiles(c, d),
                     d, c->nmax[d], c->ys, cur, c->met, c->de + 5 * d * c->NT, c->drva[d], c->NT, c->FT[d]);
    else
        LAUNCH_SWEEP(k_fd_flux_field, 1, c, d, 5, kTile, c->dblk, c->dtab, c->dlu, c->dtiles[d], ntiles(c, d), d,
                     c->nmax[d], c->ys, c->fl + 5 * d * c->NT, c->de + 5 * d * c->NT, c->drva[d], c->NT, c->FT[d]);
    return check_launch(c);
}

}  // namespace cnd
