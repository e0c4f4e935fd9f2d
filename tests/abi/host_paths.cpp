// Host paths of libdghip.so that a working GPU does not show: failing allocations and launches.  host_paths NAME runs one
// of them on the runtime of fake_hip.hpp and says what is wrong, if anything, on stderr.
#include "fake_hip.hpp"

#include "dgh.h"

#define CHECK(x)                                                                    \
    do {                                                                            \
        if (!(x)) {                                                                 \
            std::fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #x);            \
            std::exit(1);                                                           \
        }                                                                           \
    } while (0)

static dgh_ctx context() {
    dgh_ctx c = nullptr;
    CHECK(dgh_create(&c, 0) == DGH_OK);
    return c;
}

static const dgh_rhs_desc kEuler = {DGH_EQ_EULER, DGH_FLUX_LF, DGH_PREC_FP64, 0, 0, 0, 1.4};

// a failed allocation is that call's error and not the next launch's as well
static void error_is_not_kept() {
    dgh_ctx c = context();
    int m = -1, q = -1, r = -1, x = -1;
    CHECK(dgh_mesh_structured(c, 2, 3, 3, 0, 1, 0, 1, 1, 1, 0, &m) == DGH_OK);
    CHECK(dgh_field_create(c, m, 4, &q) == DGH_OK && dgh_field_create(c, m, 4, &r) == DGH_OK);
    fake::state().fail_malloc = 1;
    CHECK(dgh_field_create(c, m, 4, &x) == DGH_ERR_HIP);
    CHECK(dgh_rhs(c, m, &kEuler, q, r) == DGH_OK);
    CHECK(dgh_destroy(c) == DGH_OK);
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> all = {
        {"error_is_not_kept", error_is_not_kept},
    };
    CHECK(argc == 2 && all.count(argv[1]));
    all.at(argv[1])();
    std::puts("ok");
    return 0;
}
