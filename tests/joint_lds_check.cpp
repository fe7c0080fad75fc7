// Check of eta_zeta_joint for test_joint_lds.py: two directions whose sweeps
// fit the LDS each on their own, but not as one launch, which takes the more
// segments of the one and the partner points of the other.
#include <cstdio>

#include "../canard_amd/csrc/cnd_ctx.hpp"

using namespace cnd;

int main()
{
    const int sh = 13;   // 17-point segments, 64 pencils, eta/zeta
    const ShapeInfo &G = kShapes[sh];
    cnd_ctx c;
    const int n[3] = {20, 272, 200}, li = l_index(G.L), pi = p_index(G.P);
    for (int d = 1; d < 3; ++d) {
        c.nmax[d] = n[d];
        c.segs[li][d] = seg_count(n[d], G.L);
        c.shape[CND_KIND_FLUX][d] = sh;
        c.seg_sp[CND_KIND_FLUX][d] = round_sp(G, c.segs[li][d]);
        c.hstiles[pi][d].resize(8);
        c.classes[li][pi][d].push_back(SegClass{0, 8, c.segs[li][d], n[d]});
    }
    c.part_other[2] = true;
    const size_t eta = seg_lds_bytes(G, 1, c.seg_sp[CND_KIND_FLUX][1], n[1], false),
                 zeta = seg_lds_bytes(G, 1, c.seg_sp[CND_KIND_FLUX][2], n[2], true);
    const size_t alone = eta > zeta ? eta : zeta;
    bool ok = true;
    for (size_t lds : {alone, 2 * alone}) {
        c.lds_max = int(lds);
        if (!eta_zeta_joint(&c, CND_KIND_FLUX)) {
            ok = ok && lds == alone;
            continue;
        }
        const SegLaunches sl = seg_launches(&c, CND_KIND_FLUX, 1, 1, true);
        for (const SegLaunch &l : sl) {
            std::printf("LDS %zu: joint launch of %zu\n", lds, l.lds);
            ok = ok && l.lds <= lds && lds != alone;
        }
    }
    std::puts(ok ? "ok" : "wrong");
    return ok ? 0 : 1;
}
