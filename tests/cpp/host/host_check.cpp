// Checks of the library's host side over a runtime without a device
// (fake_hip.h), one per command-line name; see tests/test_host_side.py.
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <new>
#include <thread>

#include "../../../flipengine3d_amd/csrc/scene.h"
#include "fake_hip.h"

using namespace flipmi;
using fake::rt;

// Host allocations of this thread fail while set.
static thread_local bool t_no_host_memory = false;
void *operator new(size_t n) {
    void *p = t_no_host_memory ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

#define CHECK(c)                                            \
    do {                                                    \
        if (!(c)) {                                         \
            std::printf("line %d: %s\n", __LINE__, #c);     \
            std::exit(1);                                   \
        }                                                   \
    } while (0)
// With the two values where they differ.
#define CHECK_EQ(a, b)                                                                           \
    do {                                                                                         \
        const long long x = (long long)(a), y = (long long)(b);                                  \
        if (x != y) {                                                                            \
            std::printf("line %d: %s == %s: %lld against %lld\n", __LINE__, #a, #b, x, y);       \
            std::exit(1);                                                                        \
        }                                                                                        \
    } while (0)

// A mixed-precision projection on a store of its own.  How its two solvers end
// is set by `multigrid` and `mic0`, written over the scalars they read back.
struct Projection {
    PressureStore ps;
    PressureWork w;
    std::vector<float> grid;
    std::vector<uint8_t> flags;
    char host[kPressureStaging];
    bool multigrid = true, mic0 = true;
    hipStream_t stream = nullptr;
    Projection() {
        CHECK(hipStreamCreateWithFlags(&stream, 0) == hipSuccess);
        grid.assign(34 * 35 * 35, 0.0f);
        flags.assign(grid.size(), 0);
        w.g.I = 33; w.g.J = w.g.K = 34;
        w.g.dx = 1.0 / 32;
        w.g.invdx = 32;
        w.dt = 1.0 / 60;
        w.tol = 1e-9;
        w.acceptable = 1.0;
        w.maxiter = 100;
        w.precision = FLIPMI_PCG_MIXED;
        w.liquid = w.wU = w.wV = w.wW = w.wC = w.sU = w.sV = w.sW = grid.data();
        w.u = w.v = w.w = grid.data();
        w.vu = w.vv = w.vw = flags.data();
        rt().on_download = [this](void *dst, size_t bytes) {
            if (bytes == sizeof(MgScalars)) {
                MgScalars *sc = static_cast<MgScalars *>(dst);
                sc->bnorm = 1.0;
                sc->done = 1;
                sc->converged = multigrid;
                sc->failed = !multigrid;
            } else if (bytes == sizeof(PcgScalars)) {
                PcgScalars *sc = static_cast<PcgScalars *>(dst);
                const double one = 1.0;
                std::memcpy(&sc->absmax_bits, &one, sizeof one);
                sc->done = sc->converged = mic0;
                sc->failed = !mic0;
                sc->done = 1;
            }
        };
    }
    ~Projection() { rt().on_download = nullptr; }
    // The status a solve ends with; `first` is set to its first launch.
    int solve(size_t *first = nullptr) {
        if (first) *first = rt().launched.size();
        try {
            return run_pressure(w, ps, host, stream, nullptr).success ? FLIPMI_OK : FLIPMI_ERR_HIP;
        } catch (const StatusError &e) {
            return e.code;
        }
    }
};

// The MIC(0) iteration that takes over from multigrid does not fit: that solve
// and the next ones report it, and none runs on arrays that are not there.
static void no_room_to_fall_back() {
    Projection p;
    p.ps.alloc(p.w.g, p.stream, true, true);
    CHECK_EQ(p.solve(), FLIPMI_OK);
    {
        PressureStore slots;
        const size_t before = rt().in_use;
        slots.alloc_slots(p.w.g, p.stream, true);
        CHECK(rt().in_use - before > before);  // MIC(0)'s arrays are the larger
    }
    rt().limit = rt().in_use;
    p.multigrid = false;
    size_t first = 0;
    for (int q = 0; q < 3; q++) {
        CHECK_EQ(p.solve(&first), FLIPMI_ERR_OOM);
        CHECK(!rt().was_launched("k_reset_scalars", first) && !rt().was_launched("k_assemble", first));
        CHECK(rt().in_use <= rt().limit);
    }
    // With room again, it is solved again.
    rt().limit = ~(size_t)0;
    CHECK_EQ(p.solve(), FLIPMI_OK);
    p.multigrid = true;
    CHECK_EQ(p.solve(), FLIPMI_OK);
}

// A solve that multigrid does not converge is redone by MIC(0), and the next one
// is multigrid's again; while it keeps failing it is tried more and more rarely,
// at least once in 64 solves.
static void multigrid_again() {
    Projection p;
    p.ps.alloc(p.w.g, p.stream, true, true);
    size_t first = 0;
    auto tried = [&]() {
        CHECK_EQ(p.solve(&first), FLIPMI_OK);
        return rt().was_launched("k_mg_assemble", first);
    };
    auto redone = [&]() { return rt().was_launched("k_assemble", first); };
    CHECK(tried() && !redone());
    p.multigrid = false;
    CHECK(tried() && redone());
    p.multigrid = true;
    for (int q = 0; q < 3; q++) CHECK(tried() && !redone());
    p.multigrid = false;
    int since = 0, longest = 0, tries = 0;
    for (int q = 0; q < 400; q++) {
        if (tried()) {
            tries++;
            longest = std::max(longest, since);
            since = 0;
        } else {
            since++;
        }
        CHECK(redone());
    }
    CHECK(tries >= 7 && tries <= 12 && longest <= 64);
    // Where the count stands does not outlive the request.
    p.ps.start_over();
    p.multigrid = true;
    CHECK(tried() && !redone());
}

// Memory that a stage call left in the pool is there for every other allocation,
// and so are the blocks that a call has given back itself.
static void pool_gives_way() {
    flipmi_ctx *ctx = nullptr;
    CHECK_EQ(flipmi_ctx_create(0, &ctx), FLIPMI_OK);
    const int n = 256;
    std::vector<float> field((size_t)n * n * n, 0.0f);
    std::vector<uint8_t> valid(field.size(), 0);
    CHECK_EQ(flipmi_extrapolate(ctx, n, n, n, field.data(), valid.data(), 1), FLIPMI_OK);
    const size_t idle = rt().in_use;
    CHECK(idle > ((size_t)64 << 20));
    // Outside any stage call: all but a little of the memory is the pool's.
    rt().limit = idle + ((size_t)1 << 20);
    {
        DBuf<float> buffer;
        CHECK_EQ(buffer.alloc(field.size()), hipSuccess);
        CHECK(!buffer.scope);
        CHECK_EQ(buffer.alloc(64 * field.size()), hipErrorOutOfMemory);
        CHECK(!buffer.p && buffer.n == 0);
        CHECK_EQ(hipGetLastError(), hipSuccess);
    }
    CHECK_EQ(rt().in_use, 0);
    // Inside one: a buffer given back makes room for a larger one.
    DevicePool pool(0);
    rt().limit = 100 << 20;
    {
        hipStream_t s = nullptr;
        CHECK(hipStreamCreateWithFlags(&s, 0) == hipSuccess);
        PoolScope scope(pool, s);
        DBuf<float> a, b;
        CHECK_EQ(a.alloc(15 << 20), hipSuccess);  // 60 MiB
        a.release();
        CHECK_EQ(b.alloc(22 << 20), hipSuccess);  // 88 MiB
        CHECK_EQ(hipGetLastError(), hipSuccess);
    }
    // A block that fits exactly is had, though blocks come in steps.
    {
        pool.release();
        PoolScope scope(pool, nullptr);
        DBuf<char> c;
        CHECK_EQ(c.alloc((100 << 20) - 3), hipSuccess);
        CHECK_EQ(hipGetLastError(), hipSuccess);
    }
    pool.release();
    rt().limit = ~(size_t)0;
    CHECK_EQ(flipmi_ctx_destroy(ctx), FLIPMI_OK);
}

// Without pinned memory results come by plain copies, and the failure to get any
// is not taken for that of a later launch.
static void no_pinned_memory() {
    flipmi_ctx *ctx = nullptr;
    CHECK_EQ(flipmi_ctx_create(0, &ctx), FLIPMI_OK);
    const int n = 64;
    std::vector<float> field((size_t)n * n * n, 0.0f);
    std::vector<uint8_t> valid(field.size(), 0);
    rt().pinned_fails = true;
    for (int q = 0; q < 3; q++) {
        for (size_t c = 0; c < field.size(); c++) field[c] = (float)c;
        CHECK_EQ(flipmi_extrapolate(ctx, n, n, n, field.data(), valid.data(), 1), FLIPMI_OK);
        for (size_t c = 0; c < field.size(); c++) CHECK(field[c] == (float)c);
        CHECK_EQ(hipGetLastError(), hipSuccess);
    }
    void *page = nullptr;
    HostLink link(0);
    CHECK_EQ(link.get_page(&page), hipErrorOutOfMemory);
    CHECK_EQ(hipGetLastError(), hipSuccess);
    rt().pinned_fails = false;
    CHECK_EQ(flipmi_ctx_destroy(ctx), FLIPMI_OK);
}

// A buffer is given back without host memory to note it in: no exception leaves
// its destructor, and the device gets it.
static void give_back_without_host_memory() {
    DevicePool pool(0);
    hipStream_t s = nullptr;
    CHECK(hipStreamCreateWithFlags(&s, 0) == hipSuccess);
    bool waited = false;
    rt().on_stream_wait = [&](hipStream_t) { waited = true; };
    {
        PoolScope scope(pool, s);
        std::unique_ptr<DBuf<float>> buffer(new DBuf<float>());
        CHECK_EQ(buffer->alloc(1000), hipSuccess);
        CHECK(rt().in_use > 0);
        t_no_host_memory = true;
        buffer.reset();
        t_no_host_memory = false;
        CHECK_EQ(rt().in_use, 0);
        CHECK(waited);  // its last use may still run
    }
    rt().on_stream_wait = nullptr;
}

// While one context's kernels run, another's call begins and ends: the first
// waits for its stream until the second call has returned.
static void calls_do_not_wait_for_each_other() {
    for (int na : {16, 64, 160})
        for (int nb : {16, 64, 160}) {  // results under 256 KiB, over it, over 8 MiB
            flipmi_ctx *a = nullptr, *b = nullptr;
            CHECK_EQ(flipmi_ctx_create(0, &a), FLIPMI_OK);
            CHECK_EQ(flipmi_ctx_create(0, &b), FLIPMI_OK);
            std::mutex m;
            std::condition_variable cv;
            bool a_waits = false, b_done = false;
            rt().on_stream_wait = [&](hipStream_t s) {
                if (s != a->c.stream) return;
                std::unique_lock<std::mutex> lk(m);
                a_waits = true;
                cv.notify_all();
                CHECK(cv.wait_for(lk, std::chrono::seconds(20), [&] { return b_done; }));
            };
            auto call = [](flipmi_ctx *c, int n) {
                std::vector<float> field((size_t)n * n * n);
                std::vector<uint8_t> valid(field.size(), 0);
                for (size_t q = 0; q < field.size(); q++) field[q] = (float)(q % 4099 + n);
                CHECK_EQ(flipmi_extrapolate(c, n, n, n, field.data(), valid.data(), 1), FLIPMI_OK);
                for (size_t q = 0; q < field.size(); q++) CHECK(field[q] == (float)(q % 4099 + n));
            };
            std::thread first([&] { call(a, na); });
            {
                std::unique_lock<std::mutex> lk(m);
                CHECK(cv.wait_for(lk, std::chrono::seconds(20), [&] { return a_waits; }));
            }
            call(b, nb);
            {
                std::lock_guard<std::mutex> lk(m);
                b_done = true;
            }
            cv.notify_all();
            first.join();
            rt().on_stream_wait = nullptr;
            CHECK_EQ(flipmi_ctx_destroy(a), FLIPMI_OK);
            CHECK_EQ(flipmi_ctx_destroy(b), FLIPMI_OK);
        }
}

// Results are read from a thread whose current device is another, and nothing of
// that device gets among the context's memory.
static void another_device_is_current() {
    flipmi_ctx *ctx = nullptr;
    CHECK_EQ(flipmi_ctx_create(1, &ctx), FLIPMI_OK);
    flipmi_scene_desc d;
    flipmi_scene_desc_default(&d);
    d.isize = 24; d.jsize = d.ksize = 16;
    d.dx = 1.0 / 16;
    flipmi_scene *scene = nullptr;
    CHECK_EQ(flipmi_scene_create(ctx, &d, &scene), FLIPMI_OK);
    std::vector<float> pos(3 * 400000, 0.5f), vel(pos.size(), 0.0f), u((size_t)25 * 16 * 16);
    CHECK_EQ(flipmi_scene_load_particles(scene, pos.data(), vel.data(), (int64_t)pos.size() / 3), FLIPMI_OK);
    CHECK_EQ(flipmi_scene_initialize(scene), FLIPMI_OK);
    CHECK(hipSetDevice(0) == hipSuccess);
    const auto current = [] {
        int dev = -1;
        (void)hipGetDevice(&dev);
        return dev;
    };
    CHECK_EQ(flipmi_scene_get_particles(scene, pos.data(), vel.data()), FLIPMI_OK);
    CHECK_EQ(flipmi_scene_get_particles_range(scene, 3, 17, pos.data(), nullptr), FLIPMI_OK);
    CHECK_EQ(flipmi_scene_get_grid(scene, FLIPMI_GRID_U, u.data()), FLIPMI_OK);
    int64_t nv = 0, nt = 0;
    CHECK_EQ(flipmi_scene_get_isomesh(scene, &nv, &nt, nullptr, nullptr), FLIPMI_OK);
    CHECK_EQ(current(), 0);
    // The pool's blocks are the context's device's, whatever the call came to.
    const int n = 32;
    std::vector<float> field((size_t)n * n * n, 0.0f);
    std::vector<uint8_t> valid(field.size(), 0);
    (void)flipmi_extrapolate(ctx, n, n, n, field.data(), valid.data(), 1);
    {
        std::shared_ptr<DeviceShared> shared = DeviceShared::of(1);
        void *p = nullptr;
        size_t size = 0;
        for (size_t bytes : {sizeof(float) * field.size(), valid.size(), (size_t)1000}) {
            CHECK_EQ(shared->pool.get(bytes, &p, &size), hipSuccess);
            CHECK_EQ(fake::device_of(p), 1);
            shared->pool.put(p, size);
        }
    }
    CHECK_EQ(current(), 0);
    CHECK_EQ(flipmi_scene_destroy(scene), FLIPMI_OK);
    CHECK_EQ(flipmi_ctx_destroy(ctx), FLIPMI_OK);
}

// However many iterations the rate asks for, few batch sizes are captured.
static void few_graphs() {
    Projection p;
    p.w.graphs = &p.ps.graphs;
    p.ps.alloc(p.w.g, p.stream, true, true);
    int need = 0, looks = 0;
    rt().on_download = [&](void *dst, size_t bytes) {
        if (bytes != sizeof(MgScalars)) return;
        MgScalars *sc = static_cast<MgScalars *>(dst);
        sc->bnorm = 1.0;
        sc->tol = 1e-9;
        sc->iters = 8;
        // At the observed rate, `need` iterations more reach the tolerance.
        sc->resid = std::exp(std::log(1e-9) / (1.0 + (need - 0.5) / 8));
        sc->done = sc->converged = ++looks > 1;
    };
    for (int round = 0; round < 2; round++)
        for (need = 1; need <= 16; need++) {
            looks = 0;
            CHECK_EQ(p.solve(), FLIPMI_OK);
        }
    std::map<int, int> sizes;
    for (auto &g : p.ps.graphs.exec) sizes[g.first.first]++;
    CHECK(sizes.size() <= 8 && sizes.count(8) && sizes.count(16));
}

int main(int argc, char **argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    if (name == "no_room_to_fall_back") no_room_to_fall_back();
    else if (name == "multigrid_again") multigrid_again();
    else if (name == "pool_gives_way") pool_gives_way();
    else if (name == "no_pinned_memory") no_pinned_memory();
    else if (name == "give_back_without_host_memory") give_back_without_host_memory();
    else if (name == "calls_do_not_wait_for_each_other") calls_do_not_wait_for_each_other();
    else if (name == "another_device_is_current") another_device_is_current();
    else if (name == "few_graphs") few_graphs();
    else return 2;
    std::printf("ok\n");
    std::fflush(stdout);
    return 0;
}
