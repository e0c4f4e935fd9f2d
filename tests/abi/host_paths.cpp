// Host paths of libdghip.so that a working GPU does not show: failing allocations and launches.  host_paths NAME runs one
// of them on the runtime of fake_hip.hpp and says what is wrong, if anything, on stderr.
#include "fake_hip.hpp"

#include <chrono>
#include <condition_variable>
#include <thread>

#include "dgh.h"
#include "ensemble.hpp"
#include "stage_kernels.hpp"

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

// every stage kernel launched from now on reads and writes allocated memory
static void check_stage_operands() {
    fake::state().on_launch = [](const std::string& name, void** args) {
        if (name.find("stage_kernel") == std::string::npos && name.find("stage_sym_kernel") == std::string::npos) return;
        const dg::StageArgs& a = *static_cast<const dg::StageArgs*>(args[0]);
        CHECK(a.q_in && a.q_out);
        CHECK(fake::state().device.count(const_cast<double*>(a.q_in)) && fake::state().device.count(a.q_out));
    };
}

// a time loop whose scratch cannot be allocated: each allocation it makes fails once; the loop says so, and the next
// call runs on memory that is there
template <typename Run>
static void failing_scratch(Run run, int fields_needed) {
    for (int which = 1; which <= fields_needed; ++which) {
        dgh_ctx c = context();
        int m = -1, q = -1;
        CHECK(dgh_mesh_structured(c, 2, 3, 3, 0, 1, 0, 1, 1, 1, 0, &m) == DGH_OK);
        CHECK(dgh_field_create(c, m, 4, &q) == DGH_OK);
        check_stage_operands();
        fake::state().fail_malloc = which;
        const int before = fake::state().mallocs;
        CHECK(run(c, m, q) == DGH_ERR_HIP);
        CHECK(fake::state().mallocs == before + which);
        CHECK(fake::state().fail_malloc == 0);
        CHECK(run(c, m, q) == DGH_OK);
        CHECK(fake::state().mallocs == before + fields_needed + 1);   // no field more than the loop needs
        CHECK(run(c, m, q) == DGH_OK);
        CHECK(fake::state().mallocs == before + fields_needed + 1);
        fake::state().on_launch = nullptr;
        CHECK(dgh_destroy(c) == DGH_OK);
        CHECK(fake::state().device.empty());
    }
}

static void lserk4_scratch() {   // the residual and the second state
    failing_scratch([](dgh_ctx c, int m, int q) { return dgh_lserk4_run(c, m, &kEuler, q, 2, 1e-3, nullptr); }, 2);
}
static void ssprk2_scratch() {   // the first stage's state
    failing_scratch([](dgh_ctx c, int m, int q) { return dgh_ssprk2_run(c, m, &kEuler, nullptr, q, 2, 1e-3, nullptr); }, 1);
}

// two threads form right-hand sides of one solver with their own boundary data: from a call's copy of its data to the
// device until the call is done, nobody else writes there
static void sipg_rhs_threads() {
    dgh_ctx c = context();
    int m = -1, s = -1, f = -1, b[2];
    CHECK(dgh_mesh_structured(c, 2, 3, 3, 0, 1, 0, 1, 0, 0, DGH_BC_FIXED_VALUE, &m) == DGH_OK);
    dgh_sipg_desc d = {};
    d.maxit = 10;
    d.rtol = 1e-8;
    CHECK(dgh_sipg_create(c, m, &d, &s) == DGH_OK);
    CHECK(dgh_field_create(c, m, 1, &f) == DGH_OK);
    for (int& x : b) CHECK(dgh_field_create(c, m, 1, &x) == DGH_OK);
    const size_t n = size_t(18) * 3 * 3;
    std::mutex mu;
    std::condition_variable cv;
    std::map<void*, std::thread::id> owner;   // of a destination between the copy and the end of the call
    bool clash = false;
    fake::state().on_copy = [&](void* dst, const void*, size_t bytes, hipMemcpyKind kind) {
        if (kind != hipMemcpyHostToDevice || bytes != n * sizeof(double)) return;
        std::unique_lock<std::mutex> lock(mu);
        auto it = owner.find(dst);
        if (it != owner.end() && it->second != std::this_thread::get_id()) clash = true;
        owner[dst] = std::this_thread::get_id();
        cv.notify_all();
        cv.wait_for(lock, std::chrono::milliseconds(300), [&] { return clash; });   // the other thread's chance
    };
    fake::state().on_sync = [&] {
        std::lock_guard<std::mutex> lock(mu);
        for (auto it = owner.begin(); it != owner.end();)
            it = it->second == std::this_thread::get_id() ? owner.erase(it) : std::next(it);
    };
    std::vector<double> g[2] = {std::vector<double>(n, 1.0), std::vector<double>(n, 2.0)};
    std::vector<std::thread> t;
    for (int i = 0; i < 2; ++i)
        t.emplace_back([&, i] {
            for (int k = 0; k < 2; ++k) CHECK(dgh_sipg_rhs_neumann(c, s, f, g[i].data(), g[i].data(), b[i]) == DGH_OK);
        });
    for (auto& x : t) x.join();
    fake::state().on_copy = nullptr;
    fake::state().on_sync = nullptr;
    CHECK(!clash);
    CHECK(dgh_destroy(c) == DGH_OK);
    CHECK(fake::state().device.empty());
}

// whichever launch of an ensemble call fails, none of those before it is still running when the call returns
static void ensemble_failing_launch() {
    dgh_ctx c = context();
    const dgh_ens_desc d = {1.0, 1.0, 0.3, 0, 0};
    std::vector<dgh_ens_case> cases;
    for (int N : {2, 4, 5, 8, 3}) cases.push_back({N, 4, 4, 0, 0, 1, 1, 1.0, 0.5, 1e-3, 1e-4});
    int e = -1;
    CHECK(dgh_ensemble_create(c, &d, int(cases.size()), cases.data(), &e) == DGH_OK);
    CHECK(fake::pending() == 0);
    for (int which = 1; which <= 24; ++which) {
        fake::state().fail_launch = which;
        CHECK(dgh_ensemble_run(c, e, 1, 0, nullptr) == DGH_ERR_HIP);
        CHECK(fake::state().fail_launch == 0);
        CHECK(fake::pending() == 0);
    }
    for (int which = 1; which <= 10; ++which) {
        fake::state().fail_launch = which;
        CHECK(dgh_ensemble_rhs(c, e) == DGH_ERR_HIP);
        CHECK(fake::pending() == 0);
    }
    CHECK(dgh_ensemble_run(c, e, 1, 0, nullptr) == DGH_OK && fake::pending() == 0);
    CHECK(dgh_destroy(c) == DGH_OK);
}

// a shape that cannot be taken for want of memory leaves the ensemble as it was
static void ensemble_failing_shape() {
    dgh_ctx c = context();
    const dgh_ens_desc d = {1.0, 1.0, 0.3, 0, 0};
    std::vector<dgh_ens_case> cases;
    for (int N : {3, 5}) cases.push_back({N, 4, 4, 0, 0, 1, 1, 1.0, 0.5, 1e-3, 1e-4});
    int e = -1;
    CHECK(dgh_ensemble_create(c, &d, int(cases.size()), cases.data(), &e) == DGH_OK);
    std::vector<std::string> seen;
    bool listed = true;
    fake::state().on_launch = [&](const std::string& name, void** args) {
        const auto* a = static_cast<const dg::EnsArgs*>(args[0]);
        const auto it = fake::state().device.find(const_cast<dg::EnsItem*>(a->items));
        std::string s = name;
        for (int x : a->chunk) s += " " + std::to_string(x);
        seen.push_back(s);
        listed = listed && it != fake::state().device.end() && it->second >= size_t(a->chunk[8]) * sizeof(dg::EnsItem);
    };
    CHECK(dgh_ensemble_run(c, e, 1, 0, nullptr) == DGH_OK && listed);
    const std::vector<std::string> before = seen;
    fake::state().fail_malloc = 1;
    CHECK(dgh_ensemble_set_split(c, e, 5, 8) == DGH_ERR_HIP && fake::state().fail_malloc == 0);
    seen.clear();
    CHECK(dgh_ensemble_run(c, e, 1, 0, nullptr) == DGH_OK && listed && seen == before);
    CHECK(dgh_ensemble_set_split(c, e, 5, 8) == DGH_OK);
    seen.clear();
    CHECK(dgh_ensemble_run(c, e, 1, 0, nullptr) == DGH_OK && listed && seen != before);
    fake::state().on_launch = nullptr;
    CHECK(dgh_destroy(c) == DGH_OK);
    CHECK(fake::state().device.empty());
}

// pinned staging memory: two slots of 1 MiB, two more for every further worker of a larger transfer, given back with the
// context
static void staging_as_needed() {
    dgh_ctx c = context();
    int m = -1, f = -1, big = -1, g = -1;
    CHECK(dgh_mesh_structured(c, 2, 3, 3, 0, 1, 0, 1, 1, 1, 0, &m) == DGH_OK);
    CHECK(dgh_field_create(c, m, 4, &f) == DGH_OK);
    CHECK(fake::state().pinned_bytes == 0);
    std::vector<double> a(size_t(18) * 6 * 4, 1.0);
    CHECK(dgh_field_upload(c, f, a.data()) == DGH_OK && dgh_field_download(c, f, a.data()) == DGH_OK);
    CHECK(fake::state().pinned_bytes == size_t(2) << 20);
    CHECK(dgh_mesh_structured(c, 8, 64, 32, 0, 1, 0, 1, 1, 1, 0, &big) == DGH_OK);
    CHECK(dgh_field_create(c, big, 4, &g) == DGH_OK);
    std::vector<double> b(size_t(4096) * 45 * 4, 1.0);
    CHECK(dgh_field_upload(c, g, b.data()) == DGH_OK);
    CHECK(fake::state().pinned_bytes == size_t(2) << 20);
    for (int n : {2, 16}) {   // workers: one for every 8 MiB, at most eight
        const int K = 2 * 64 * 16 * n;
        CHECK(dgh_mesh_structured(c, 8, 64, 16 * n, 0, 1, 0, 1, 1, 1, 0, &big) == DGH_OK);
        CHECK(dgh_field_create(c, big, 4, &g) == DGH_OK);
        b.assign(size_t(K) * 45 * 4, 1.0);
        CHECK(dgh_field_upload(c, g, b.data()) == DGH_OK);
        const size_t workers = std::max<size_t>(1, std::min<size_t>(8, b.size() * sizeof(double) >> 23));
        CHECK(fake::state().pinned_bytes == 2 * workers << 20);
    }
    CHECK(dgh_field_download(c, f, a.data()) == DGH_OK);
    CHECK(fake::state().pinned.size() == 1);
    CHECK(dgh_destroy(c) == DGH_OK);
    CHECK(fake::state().pinned.empty());
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> all = {
        {"error_is_not_kept", error_is_not_kept},
        {"lserk4_scratch", lserk4_scratch},
        {"ssprk2_scratch", ssprk2_scratch},
        {"sipg_rhs_threads", sipg_rhs_threads},
        {"ensemble_failing_launch", ensemble_failing_launch},
        {"ensemble_failing_shape", ensemble_failing_shape},
        {"staging_as_needed", staging_as_needed},
    };
    CHECK(argc == 2 && all.count(argv[1]));
    all.at(argv[1])();
    std::puts("ok");
    return 0;
}
