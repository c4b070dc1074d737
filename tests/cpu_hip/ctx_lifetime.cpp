// A lattice outlives the context it was made on: every call that does not ask
// for the device itself goes on working (the C++ layer's set_device replaces
// the context while States may be alive).  Under AddressSanitizer against the
// CPU model of the HIP runtime; test infrastructure.
#include <cstdio>
#include <vector>

#include "chemsim.h"

static int failures = 0;
#define OK(call)                                                                    \
    do {                                                                            \
        if ((call) != CS_OK) {                                                      \
            std::fprintf(stderr, "FAILED %s: %s\n", #call, cs_last_error());        \
            ++failures;                                                             \
        }                                                                           \
    } while (0)

int main()
{
    const int w = 70, h = 50;
    std::vector<float> a((size_t)w * h, 1.0f), ux((size_t)w * h, 0.0f), uy(ux);
    std::vector<double> d((size_t)w * h);
    for (int storage = CS_F32; storage <= CS_F32DEV; ++storage) {
        cs_ctx* ctx = nullptr;
        cs_lattice *l = nullptr, *other = nullptr;
        OK(cs_ctx_create(0, &ctx));
        OK(cs_lattice_create(ctx, w, h, storage, &l));
        OK(cs_lattice_create(ctx, w, h, storage, &other));
        OK(cs_lattice_velocity(l, ux.data(), uy.data()));
        OK(cs_ctx_destroy(ctx));
        int k = 0;
        OK(cs_lattice_temporal_steps(l, &k));
        OK(cs_lattice_step(l, 21));
        OK(cs_lattice_density(l, a.data()));
        OK(cs_lattice_velocity(other, ux.data(), uy.data()));
        OK(cs_lattice_destroy(l));
        OK(cs_lattice_moments_f64(other, d.data(), d.data(), nullptr));
        OK(cs_lattice_destroy(other));
    }
    if (failures == 0) std::printf("lattices after their context: ok\n");
    return failures != 0;
}
