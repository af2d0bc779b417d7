// The level-0 inverse when its device workspace cannot be had: the host elimination takes its place.  This
// program's hipMalloc stands before the HIP runtime's and refuses allocations from a given size on.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <vector>

#include "cirrus_amg.h"

namespace {
size_t refuse_from = ~size_t(0);
int refused = 0;
}  // namespace

extern "C" int hipMalloc(void** p, size_t n)
{
    static auto real = reinterpret_cast<int (*)(void**, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    if (n >= refuse_from) {
        ++refused;
        *p = nullptr;
        return 2;   // hipErrorOutOfMemory
    }
    return real(p, n);
}

#define CHECK(call)                                                                               \
    do {                                                                                          \
        if ((call) != CMG_OK) {                                                                   \
            std::printf("line %d: %s\n", __LINE__, cmg_last_error());                            \
            return 1;                                                                             \
        }                                                                                         \
    } while (0)

int main()
{
    // one tile with 437 unknowns: the two work matrices are 448 x 448 FP64 each, the inverse 437 x 437
    const uint32_t log2[1] = {4};
    cmg_grid* g = nullptr;
    CHECK(cmg_grid_create(0.125f, 1, log2, &g));
    CHECK(cmg_grid_set_tile(g, 0, 0, 0, 0, CMG_LEAF));
    CHECK(cmg_grid_rebuild(g));
    CHECK(cmg_grid_finalize(g));
    std::vector<uint8_t> types(512, CMG_INTERIOR);
    for (int i = 0; i < 75; ++i) types[size_t(i) * 97 % 512] = CMG_DIRICHLET;
    CHECK(cmg_grid_set_cell_types(g, types.data()));
    CHECK(cmg_prepare_types_and_coeffs(g, 11, 0.5f));
    CHECK(cmg_rhs_uniform(g, 1, 9, 0));
    std::vector<float> x[2];
    for (int k = 0; k < 2; ++k) {
        cmg_solver* s = nullptr;
        CHECK(cmg_solver_create(g, 11, 0.5f, 1.0f, 1.0f, &s));
        cmg_solve_opts o;
        cmg_solve_opts_default(&o);
        o.cycle = CMG_CYCLE_FAS_V;
        o.smoother = CMG_SMOOTH_JACOBI;
        o.coarsest_direct = 1;
        refuse_from = k ? size_t(2) * 448 * 448 * 8 : ~size_t(0);
        CHECK(cmg_op_cycle(s, &o, 4, 1, 3));
        refuse_from = ~size_t(0);
        x[k].resize(512);
        CHECK(cmg_grid_get_channel(g, 4, x[k].data()));
        cmg_solver_destroy(s);
    }
    cmg_grid_destroy(g);
    float top = 0, diff = 0;
    for (int v = 0; v < 512; ++v) {
        top = std::fmax(top, std::fabs(x[0][v]));
        diff = std::fmax(diff, std::fabs(x[0][v] - x[1][v]));
    }
    std::printf("refused %d, largest value %g, largest difference %g\n", refused, top, diff);
    // one FP32 rounding of two FP64 solutions
    if (refused < 1 || !(top > 0) || !(diff <= top * 0x1p-23f)) return 1;
    std::printf("inverse fallback OK\n");
    return 0;
}
