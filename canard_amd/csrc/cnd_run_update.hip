// The last flux sweep of a stage (direction fuse_dir) fused with the
// RK update.
#include "cnd_ctx.hpp"

namespace cnd {

int run_flux_update(cnd_ctx *c, int nk, double *qa)
{
    LAUNCH_SEG((k_seg_flux_update<G>), c, seg_launches(c, CND_KIND_FLUX, c->fuse_dir, 1), 5, 1, c->dinst, c->fl, c->de,
               c->qo, c->met, qa, ends3(c), c->NT, nk);
    return check_launch(c);
}

}  // namespace cnd
