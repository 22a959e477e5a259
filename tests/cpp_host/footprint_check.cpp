// What a hierarchy of constant coefficients takes against opf_gmg_footprint, by which the server admits
// requests (no GPU): while it is built and afterwards, with coarsest levels of a few cells to 1024.
#include <array>
#include <cstdio>

#include "gmg.hpp"
#include "hip_standins.hpp"
#include "opf_internal.hpp"

using namespace opf;

int main() {
    opf_ctx ctx{};
    for (auto n : {std::array{64, 64, 1}, {256, 256, 1}, {160, 100, 1}, {640, 400, 1}, {62, 62, 1}, {33, 31, 1}, {128, 128, 1},
                   {320, 200, 1}, {20, 20, 20}, {64, 64, 64}, {40, 36, 28}, {80, 72, 56}, {32, 32, 1}, {496, 528, 1}})
        for (int precision : {OPF_PREC_FP64, OPF_PREC_MIXED})
            for (int slots : {1, 8}) {
                opf_poisson_desc d{};
                d.dim = n[2] > 1 ? 3 : 2;
                GLevelHost L{};
                L.N = 1;
                for (int q = 0; q < 3; ++q) {
                    d.n[q] = L.n[q] = n[q];
                    d.h[q] = 1.0;
                    L.a[q] = q < d.dim;
                    L.N *= n[q];
                    for (int s = 0; s < 2; ++s) d.bc[q][s] = OPF_BC_DIRC;
                }
                const int per[3] = {0, 0, 0};
                const double alpha[3][2] = {{-1, -1}, {-1, -1}, {-1, -1}};
                Hierarchy H;
                held_bytes = peak_bytes = 0;
                if (gmg_build(&ctx, H, L, per, alpha, precision, slots) != OPF_OK) return std::printf("build\n"), 1;
                const size_t most = hier_footprint(&d, precision, slots), one = opf_gmg_footprint(&d, precision);
                if (held_bytes > most || peak_bytes > most)
                    return std::printf("%d x %d x %d, %d slots: %zu, in the build %zu, of %zu\n", n[0], n[1], n[2], slots,
                                       held_bytes, peak_bytes, most), 1;
                if (slots == 1 && one != most) return std::printf("one slot\n"), 1;
                if (H.cwork) return std::printf("scratch kept\n"), 1;
                if (H.bytes > held_bytes) return std::printf("counted %zu of %zu\n", H.bytes, held_bytes), 1;
                gmg_free(H);
            }
    std::printf("passed\n");
    return 0;
}
