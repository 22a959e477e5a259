// A multigrid hierarchy whose build runs out of device memory, then builds again (no GPU: this program
// stands in for the HIP calls of the library). At every
// allocation in turn: the failing build reports it, the next one leaves a hierarchy with all of its
// buffers, and freeing it leaves none behind.
#include <cstdio>

#include "gmg.hpp"
#include "hip_standins.hpp"
#include "opf_internal.hpp"

using namespace opf;

static bool whole(const Hierarchy& H) {
    bool ok = H.cinv && H.r && H.z && H.p[0] && H.p[1] && H.q && H.e && H.r64 && H.part && H.scal && H.hscal && H.mk;
    ok &= H.cwork || !H.var;  // a variable operator is inverted again at the next solve
    for (size_t l = 0; l < H.dev.size(); ++l) {
        ok &= H.dev[l].t && (l == 0 || (H.dev[l].x && H.dev[l].b));
        if (H.var) ok &= H.dev[l].sg64 && H.dev[l].af64[0] && (H.precision != OPF_PREC_MIXED || H.dev[l].sg32);
    }
    return ok;
}

int main() {
    opf_ctx ctx{};
    const int per[3] = {0, 0, 0};
    const double alpha[3][2] = {{-1, -1}, {-1, -1}, {-1, -1}};
    for (bool var : {true, false})
        for (int precision : {OPF_PREC_FP64, OPF_PREC_MIXED}) {
            DevLevel fine;
            fine.n[0] = 160, fine.n[1] = 100;
            fine.N = 16000;
            fine.var = var;
            fine.a[0] = fine.a[1] = 1.0;
            for (int d = 0; d < 2; ++d) hipMalloc((void**)&fine.af[d], sizeof(double) * level_face_count(fine.n, d));
            hipMalloc((void**)&fine.sg, sizeof(double) * fine.N);
            const size_t before = live.size();
            Hierarchy H;
            fail_at = -1;
            calls = 0;
            if (gmg_build_dev(&ctx, H, fine, per, alpha, precision) != OPF_OK || !whole(H)) return std::printf("first build\n"), 1;
            const long long n = calls;
            const size_t held = live.size();
            if (gmg_build_dev(&ctx, H, fine, per, alpha, precision) != OPF_OK || calls != n || live.size() != held)
                return std::printf("a rebuild keeps the buffers\n"), 1;
            gmg_free(H);
            if (live.size() != before) return std::printf("buffers left behind\n"), 1;
            for (long long k = 0; k < n; ++k) {
                Hierarchy G;
                fail_at = k;
                calls = 0;
                if (gmg_build_dev(&ctx, G, fine, per, alpha, precision) == OPF_OK) return std::printf("allocation %lld\n", k), 1;
                fail_at = -1;
                if (gmg_build_dev(&ctx, G, fine, per, alpha, precision) != OPF_OK || !whole(G) || live.size() != held)
                    return std::printf("var %d precision %d: after allocation %lld of %lld failed: %zu of %zu buffers\n", var,
                                       precision, k, n, live.size(), held), 1;
                gmg_free(G);
                if (live.size() != before) return std::printf("buffers left behind after %lld\n", k), 1;
            }
            for (int d = 0; d < 2; ++d) hipFree(fine.af[d]);
            hipFree(fine.sg);
        }
    std::printf("passed\n");
    return 0;
}
