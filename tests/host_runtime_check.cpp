// What a handle keeps alive, and for how long: the engine's host code on a stand-in runtime
// (host_runtime.h), under AddressSanitizer. Built and run by tests/test_host_runtime.py, one check a run:
// host_runtime_check <check>.
#include <cmath>
#include <random>

#include "host_runtime.h"

namespace {

using rt::Launch;

// Inputs of a small run: isotropic, per-axis or exponential; every source point is also a sensor, so that
// the records hold the signals whatever the stencils do.
struct Inputs {
    fw_desc d{};
    std::map<std::string, std::vector<float>> f;
    std::map<std::string, std::vector<int32_t>> i;
    int64_t cells() const { return d.nx * d.ny * d.nz; }
};

Inputs inputs(int ndim, int64_t nx, int64_t ny, int64_t nz, int64_t nt, int isotropic = 1, int model = 0, int sound_speeds = 3) {
    Inputs in;
    fw_desc& d = in.d;
    d.abi_version = FW_ABI_VERSION;
    d.ndim = ndim;
    d.isotropic = isotropic;
    d.attenuation_model = model;
    d.n_relax = 2;
    d.nx = nx, d.ny = ny, d.nz = ndim == 3 ? nz : 1;
    d.nt = nt;
    d.dx = d.dy = d.dz = 4.3e-5;
    d.dt = 1.1e-8;
    d.c0 = 1540;
    d.modt = 2;
    d.ndmap = sound_speeds;
    const int64_t n = in.cells();
    std::mt19937 rng(5);
    auto map = [&](const std::string& name, float lo, float step) {  // a few values in patches
        std::vector<float> v((size_t)n);
        for (int64_t c = 0; c < n; ++c) v[(size_t)c] = lo + step * (float)(c * 3 / n);
        in.f[name] = v;
    };
    map("K", 2e9f, 1e8f);
    map("rho", 1000.f, 10.f);
    const char *av[3] = {"u", "w", "v"}, *ap[3] = {"x", "y", "z"};
    if (model == 1) map("a_exp", 0.9f, 0.01f);
    for (int a = 0; a < (isotropic ? 1 : ndim) && model == 0; ++a)
        for (const char* x : {av[a], ap[a]}) {
            map(std::string("kappa") + x, 1.f, 0.1f);
            for (const char* nu : {"1", "2"}) {
                map(std::string("apml") + x + nu, -0.1f, 0.01f);
                map(std::string("bpml") + x + nu, 0.8f, 0.01f);
            }
        }
    in.f["dmap"].assign((size_t)(18 * d.ndmap), 0.1f);
    auto& dc = in.i["dcmap"];
    for (int64_t c = 0; c < n; ++c) dc.push_back((int32_t)(c * sound_speeds / n));
    auto& src = in.i["icc"];
    const int64_t dims[3] = {nx, ny, nz};
    d.ncoords = 9;
    for (int64_t q = 0; q < d.ncoords; ++q)
        for (int a = 0; a < ndim; ++a) src.push_back((int32_t)(a == 0 ? 8 + q % (nx - 16) : 8 + (7 * q) % (dims[a] - 16)));
    in.i["outc"] = src;
    d.ncoordsout = d.ncoords;
    d.ntic = nt;
    auto& sig = in.f["icmat"];
    for (int64_t k = 0; k < d.ncoords * d.ntic; ++k) sig.push_back((float)(rng() % 1000) + 1.f);
    return in;
}

fw_sim* make(const Inputs& in) {
    fw_sim* s = nullptr;
    CHECK(fw_sim_create(&in.d, 0, &s) == FW_OK);
    for (const auto& m : in.f) CHECK(fw_sim_upload(s, m.first.c_str(), m.second.data(), m.second.size() * 4) == FW_OK);
    for (const auto& m : in.i) CHECK(fw_sim_upload(s, m.first.c_str(), m.second.data(), m.second.size() * 4) == FW_OK);
    return s;
}

void pin(fw_sim* s, int variant, int width, int chunk) {
    for (int kind = 0; kind < 2; ++kind) CHECK(fw_sim_set_kernel_config(s, kind, variant, width, chunk) == FW_OK);
}

// run `steps` from rest; the records are the signals
void run_and_check(fw_sim* s, const Inputs& in, int64_t steps) {
    CHECK(fw_sim_reset(s) == FW_OK);
    const int rc = fw_sim_run(s, steps);
    CHECK(rc == FW_OK);
    if (rc != FW_OK) {
        std::fprintf(stderr, "run: %s\n", fw_last_error());
        return;
    }
    const int64_t rows = (steps + in.d.modt - 1) / in.d.modt;
    std::vector<float> rec((size_t)(rows * in.d.ncoordsout));
    CHECK(fw_sim_download_sensors(s, rec.data(), rec.size() * 4) == FW_OK);
    for (int64_t r = 0; r < rows; ++r)
        for (int64_t q = 0; q < in.d.ncoordsout; ++q)
            CHECK(rec[(size_t)(r * in.d.ncoordsout + q)] == in.f.at("icmat")[(size_t)(q * in.d.ntic + r * in.d.modt)]);
}

// An adjoint made on a handle that has run from a captured graph: the graph's launches hold the address of
// the point table that the adjoint's kernels replace.
void graph_then_adjoint() {
    struct Pin {
        int ndim, variant, width, chunk;
    };
    for (const Pin& p : {Pin{2, 1, 64, 5}, Pin{2, 2, 256, 32}, Pin{2, 0, 0, 0}, Pin{3, 0, 0, 0}, Pin{3, 5, 32, 1}}) {
        const Inputs in = inputs(p.ndim, 40, 36, 44, 24);
        fw_sim* s = make(in);
        pin(s, p.variant, p.width, p.chunk);
        CHECK(fw_sim_set_graph_steps(s, 4) == FW_OK);
        run_and_check(s, in, 10);
        fw_adj* a = nullptr;
        CHECK(fw_adj_create(s, 8, &a) == FW_OK);
        run_and_check(s, in, 10);
        run_and_check(s, in, 24);
        CHECK(fw_adj_destroy(a) == FW_OK && fw_sim_destroy(s) == FW_OK);
    }
}

// A handle of no steps has no records: choosing its kernels writes none.
void no_records() {
    for (int ndim : {2, 3}) {
        Inputs in = inputs(ndim, 40, 36, 44, 6);
        in.d.nt = 0;
        fw_sim* s = make(in);
        int32_t v, w, c;
        CHECK(fw_sim_kernel_config(s, 1, &v, &w, &c) == FW_OK);
        CHECK(fw_sim_run(s, 0) == FW_OK && fw_sim_run(s, 1) == FW_ERR_INVALID);
        CHECK(fw_sim_destroy(s) == FW_OK);
    }
}

// Bricks need codes: a brick handle that replays captured steps runs on after its codes are gone (switched
// off; one axis with a map of its own), and with bricks again when they are back.
void graph_without_codes() {
    for (int isotropic : {1, 0}) {
        const Inputs in = inputs(3, 24, 26, 44, 24, isotropic);
        fw_sim* s = make(in);
        pin(s, 5, 32, 1);
        CHECK(fw_sim_set_graph_steps(s, 4) == FW_OK);
        run_and_check(s, in, 10);
        CHECK(fw_sim_set_relaxation_codes(s, 0) == FW_OK);
        run_and_check(s, in, 10);
        CHECK(fw_sim_set_relaxation_codes(s, 1) == FW_OK);
        run_and_check(s, in, 10);
        const char* last = isotropic ? "bpmlx2" : "bpmlz2";
        std::vector<float> own = in.f.at(last);
        for (size_t c = 0; c < own.size(); ++c) own[c] = isotropic ? 1e-6f * (float)c : own[c] * 0.5f;  // too many codes
        CHECK(fw_sim_upload(s, last, own.data(), own.size() * 4) == FW_OK);
        run_and_check(s, in, 10);
        CHECK(fw_sim_upload(s, last, in.f.at(last).data(), own.size() * 4) == FW_OK);
        rt::log.clear();
        rt::keep_log = true;
        run_and_check(s, in, 10);
        rt::keep_log = false;
        int bricks = 0;
        for (const Launch& l : rt::log) bricks += l.is("k_pressure_brick");
        CHECK(bricks == 10);
        CHECK(fw_sim_destroy(s) == FW_OK);
    }
}

std::string config(fw_sim* s, int kind) {
    int32_t v = -1, w = 0, c = 0;
    CHECK(fw_sim_kernel_config(s, kind, &v, &w, &c) == FW_OK);
    return std::to_string(v) + ":" + std::to_string(w) + ":" + std::to_string(c);
}

// The kernels of a brick handle whose codes go away: the fastest of the others where they were timed, the
// stated default where they were not, the per-cell ones (which write the tape) for an adjoint; the bricks
// again with the codes.
void kernels_without_codes() {
    rt::cost = [](const Launch& l) {
        if (l.is("k_velocity_brick") || l.is("k_pressure_brick")) return 10.0;
        if (l.is("k_velocity_pipe3d")) return 20.0 + std::abs(l.arg<int>(1) - 48) + (l.name.find("<16, ") != std::string::npos ? 3 : 0);
        if (l.is("k_pressure_pipe3d")) return 20.0 + std::abs(l.arg<int>(1) - 16) + (l.name.find("<16, ") != std::string::npos ? 0 : 3);
        return l.is("k_boundary") ? 1.0 : 100.0;
    };
    const Inputs in = inputs(3, 24, 26, 44, 24);
    const std::vector<float> zero((size_t)in.cells(), 0.f);
    for (int how = 0; how < 3; ++how) {  // timed, a field set before the first run, bound to an adjoint
        fw_sim* s = make(in);
        if (how == 1) CHECK(fw_sim_set_field(s, "p", zero.data(), zero.size() * 4) == FW_OK);
        fw_adj* a = nullptr;
        if (how == 2) pin(s, 5, 32, 1);  // (few bricks: not the adjoint's own choice)
        if (how == 2) CHECK(fw_adj_create(s, 8, &a) == FW_OK);
        for (int round = 0; round < 2; ++round) {
            run_and_check(s, in, 10);
            for (int kind = 0; kind < 2; ++kind) CHECK(config(s, kind).compare(0, 5, "5:32:") == 0);
            CHECK(fw_sim_set_relaxation_codes(s, 0) == FW_OK);
            rt::log.clear();
            rt::keep_log = true;
            run_and_check(s, in, 10);
            rt::keep_log = false;
            int march = 0, cell = 0;
            for (const Launch& l : rt::log) {
                march += l.is("k_velocity_pipe3d") || l.is("k_pressure_pipe3d") || l.is("k_velocity_3d") || l.is("k_pressure_3d");
                cell += l.is("k_velocity_cell") || l.is("k_pressure_cell");
            }
            CHECK(march == (how == 2 ? 0 : 20) && cell == (how == 2 ? 20 : 0));
            const std::string v = config(s, 0), p = config(s, 1);
            if (how == 0) CHECK((v == "3:512:48" || v == "4:512:48") && (p == "3:1024:16" || p == "4:1024:16"));
            if (how == 1) CHECK(v == "1:512:8" && p == "1:512:8");
            if (how == 2) CHECK(v[0] == '0' && p[0] == '0');
            CHECK(fw_sim_set_relaxation_codes(s, 1) == FW_OK);
        }
        CHECK(fw_adj_destroy(a) == FW_OK && fw_sim_destroy(s) == FW_OK);
    }
}

// A process whose launches cost what `us` says; the code of each of the engine's source files takes 3 ms
// to load, at the first use of one of its kernels.
template <class F>
void launch_costs(std::set<std::string>* loaded, const F& us) {
    loaded->clear();
    rt::load = [loaded](const std::string& n) {
        const char* files[] = {"brick", "pipe3d", "_tile", "_2d", "_3d", "code"};
        std::string file = "cell";
        for (const char* f : files)
            if (n.find(f) != std::string::npos) {
                file = f;
                break;
            }
        return loaded->insert(file).second ? 3000.0 : 0.0;
    };
    rt::cost = us;
}

// The kernels that timing keeps are the fastest of the candidates, whatever a first launch costs.
void timing() {
    std::set<std::string> loaded;
    const Inputs in = inputs(3, 24, 26, 44, 4);
    auto kernels = [&](const Inputs& i) {
        fw_sim* s = make(i);
        const std::string c = config(s, 0) + " " + config(s, 1);
        CHECK(fw_sim_destroy(s) == FW_OK);
        return c;
    };
    // long kernels: the bricks' first order, and the last of the marching families
    launch_costs(&loaded, [](const Launch& l) {
        if (l.is("k_velocity_brick")) return l.arg<bool>(3) ? 900.0 : 835.0;
        if (l.is("k_pressure_brick")) return l.arg<bool>(3) ? 857.0 : 880.0;
        if (l.is("k_velocity_pipe3d")) return 893.0 + std::abs(l.arg<int>(1) - 48);
        if (l.is("k_pressure_pipe3d")) return l.name.find("<16, ") != std::string::npos && l.arg<int>(1) == 8 ? 839.0 : 950.0;
        return l.is("k_boundary") ? 4.0 : 2000.0;
    });
    CHECK(kernels(in) == "5:32:0 3:1024:8");
    CHECK(kernels(in) == "5:32:0 3:1024:8");  // a later handle of the process
    // short ones
    launch_costs(&loaded, [](const Launch& l) {
        if (l.is("k_velocity_brick")) return l.arg<bool>(3) ? 21.0 : 22.0;
        if (l.is("k_pressure_brick")) return l.arg<bool>(3) ? 23.0 : 22.0;
        return l.is("k_boundary") ? 4.0 : 25.0;
    });
    CHECK(kernels(in) == "5:32:1 5:32:0");
    // a long kernel whose first timed launch is short by 5 %: the fastest two are launched again
    std::map<std::string, int> seen;
    launch_costs(&loaded, [&seen](const Launch& l) {
        const bool v = l.is("k_velocity_brick"), p = l.is("k_pressure_brick");
        if (!v && !p) return l.is("k_boundary") ? 4.0 : 3000.0;
        const bool order = l.arg<bool>(3), slow = order == p;
        const bool odd = slow && ++seen[l.name] == 1;
        return slow ? odd ? 965.0 : 1015.0 : 1000.0;
    });
    CHECK(kernels(in) == "5:32:1 5:32:0");
    // points that no pressure launch takes: every family makes a boundary launch, and none is charged for it
    Inputs many = in;
    many.i["outc"].clear();
    many.d.ncoordsout = (int64_t(1) << 18) + 1;
    for (int64_t q = 0; q < 3 * many.d.ncoordsout; ++q) many.i["outc"].push_back(9);
    auto marching = [](const Launch& l) {
        if (l.is("k_velocity_brick") || l.is("k_pressure_brick")) return 103.0;
        if (l.is("k_velocity_pipe3d") || l.is("k_pressure_pipe3d")) return l.arg<int>(1) == 16 ? 100.0 : 110.0;
        return l.is("k_boundary") ? 10.0 : 200.0;
    };
    launch_costs(&loaded, marching);
    CHECK(kernels(many) == "3:512:16 3:512:16");
    launch_costs(&loaded, marching);
    CHECK(kernels(in) == "3:512:16 5:32:0");  // points that a pressure launch takes
}

// A set of per-axis maps uploaded again: the maps are compared and coded once, by the next run, and until then
// nothing of the old codes is used. One axis with a map of its own is found, also by an adjoint's run.
void per_axis_uploads() {
    for (int ndim : {2, 3}) {
        const Inputs in = inputs(ndim, 24, 28, 44, 24, 0);
        fw_sim* s = make(in);
        auto again = [&](const char* own) {
            for (const auto& m : in.f) {
                const bool map = m.first.compare(0, 5, "kappa") == 0 || m.first.compare(1, 3, "pml") == 0;
                if (!map) continue;
                std::vector<float> v = m.second;
                for (size_t c = 0; own && m.first == own && c < v.size(); ++c) v[c] *= 0.5f;
                CHECK(fw_sim_upload(s, m.first.c_str(), v.data(), v.size() * 4) == FW_OK);
            }
        };
        auto count = [&](const char* kernel) {
            int n = 0;
            for (const Launch& l : rt::log) n += l.is(kernel) && !l.is("k_maps_differ_tail");
            return n;
        };
        CHECK(fw_sim_set_graph_steps(s, 4) == FW_OK);
        run_and_check(s, in, 10);
        fw_adj* a = nullptr;
        const std::vector<float> w(in.d.ncoordsout * 12, 1.f);
        std::vector<float> gk((size_t)in.cells()), gr((size_t)in.cells());
        auto gradient = [&] {
            CHECK(fw_adj_forward(a) == FW_OK);
            CHECK(fw_adj_backward(a, w.data(), w.size() * 4, gk.data(), gr.data(), gk.size() * 4) == FW_OK);
        };
        for (const char* own : {(const char*)nullptr, ndim == 2 ? "bpmly2" : "bpmlz2", (const char*)nullptr}) {
            rt::log.clear();
            rt::keep_log = true;
            again(own);
            CHECK(count("k_maps_differ") == 0 && count("k_code_insert") == 0);
            if (a) gradient();
            run_and_check(s, in, 10);
            rt::keep_log = false;
            CHECK(count("k_maps_differ") == 1 && count("k_code_insert") == (own ? 0 : 1));
            if (!a) CHECK(fw_adj_create(s, 8, &a) == FW_OK);
            gradient();
            again(nullptr);
            CHECK(fw_adj_backward(a, w.data(), w.size() * 4, gk.data(), gr.data(), gk.size() * 4) == FW_OK);
        }
        CHECK(fw_adj_destroy(a) == FW_OK && fw_sim_destroy(s) == FW_OK);
    }
}

// Gradients with every list that an adjoint builds (sensors on planes, on sources, on release points and
// twice on a voxel), destroyed after its simulation's handle, before it, and with the runtime's ordinary
// allocations in place of the stream-ordered ones.
void adjoint_lifetimes() {
    struct Case {
        int ndim, model, isotropic;
        int64_t nx, ny, nz, nt, every;
    };
    for (const Case& c : {Case{3, 0, 1, 136, 120, 112, 4, 4}, Case{3, 0, 1, 21, 25, 41, 9, 4}, Case{3, 1, 1, 18, 33, 43, 9, 0},
                          Case{3, 0, 0, 21, 25, 41, 9, 9}, Case{2, 0, 1, 25, 81, 1, 9, 4}, Case{2, 0, 0, 67, 212, 1, 9, 0},
                          Case{2, 1, 1, 21, 26, 1, 9, 1}}) {
        Inputs in = inputs(c.ndim, c.nx, c.ny, c.nz, c.nt, c.isotropic, c.model);
        auto& out = in.i["outc"];
        auto& air = in.i["icczero"];
        const int64_t dims[3] = {c.nx, c.ny, in.d.nz};
        auto plane = [&](int axis) {
            for (int64_t i = 0; i < dims[0]; ++i)
                for (int64_t j = 0; j < dims[1]; ++j)
                    for (int64_t k = 0; k < dims[2]; ++k) {
                        const int64_t x[3] = {i, j, k};
                        if (x[axis] != dims[axis] / 2) continue;
                        for (int a = 0; a < c.ndim; ++a) out.push_back((int32_t)x[a]);
                    }
        };
        for (int a = 0; a < c.ndim; ++a) plane(a);
        for (int q = 0; q < 12 * c.ndim; ++q) air.push_back((int32_t)(q % c.ndim == 0 ? q % 2 ? dims[0] - 1 : 3 : 0));  // corners
        for (int q = 0; q < 3 * c.ndim; ++q) air.push_back(in.i["icc"][(size_t)q]);
        in.d.ncoordszero = (int64_t)air.size() / c.ndim;
        in.d.ncoordsout = (int64_t)out.size() / c.ndim;
        for (int order = 0; order < 3; ++order) {
            rt::async_fails = order == 2;
            fw_sim* s = make(in);
            fw_adj* a = nullptr;
            CHECK(fw_adj_create(s, c.every, &a) == FW_OK);
            const std::vector<float> w((size_t)(in.d.ncoordsout * ((c.nt + 1) / 2)), 1.f);
            std::vector<float> gk((size_t)in.cells()), gr((size_t)in.cells());
            for (int pass = 0; pass < 2; ++pass) {
                CHECK(fw_adj_forward(a) == FW_OK);
                CHECK(fw_adj_backward(a, w.data(), w.size() * 4, gk.data(), gr.data(), gk.size() * 4) == FW_OK);
            }
            if (order == 1) {
                CHECK(fw_sim_destroy(s) == FW_OK);
                CHECK(fw_adj_forward(a) == FW_ERR_STATE);
                CHECK(fw_adj_backward(a, w.data(), w.size() * 4, gk.data(), gr.data(), gk.size() * 4) == FW_ERR_STATE);
                CHECK(fw_adj_destroy(a) == FW_OK);
            } else {
                CHECK(fw_adj_destroy(a) == FW_OK);
                CHECK(fw_sim_destroy(s) == FW_OK);
            }
            rt::async_fails = false;
        }
    }
}

// The kernels of an adjoint's taped steps: bricks from 160 of them on, else the per-cell kernels; a pinned
// family that writes the tape stays.
void taped_kernels() {
    struct Case {
        int64_t nx, ny, nz;
        int variant;
    };
    for (int model : {0, 1})
        for (const Case& c : {Case{24, 26, 44, 0}, Case{64, 64, 64, 0}, Case{68, 66, 64, 5}})
            for (bool pinned : {false, true}) {
                const Inputs in = inputs(3, c.nx, c.ny, c.nz, 4, 1, model);
                fw_sim* s = make(in);
                if (pinned) pin(s, 5, 32, 0);
                fw_adj* a = nullptr;
                CHECK(fw_adj_create(s, 2, &a) == FW_OK);
                const int want = pinned ? 5 : c.variant;
                for (int kind = 0; kind < 2; ++kind) CHECK(config(s, kind)[0] == '0' + want);
                CHECK(fw_adj_forward(a) == FW_OK);
                CHECK(fw_adj_destroy(a) == FW_OK && fw_sim_destroy(s) == FW_OK);
            }
}

struct Check {
    const char* name;
    void (*run)();
};
const Check checks[] = {
    {"graph_then_adjoint", graph_then_adjoint},
    {"no_records", no_records},
    {"graph_without_codes", graph_without_codes},
    {"kernels_without_codes", kernels_without_codes},
    {"timing", timing},
    {"per_axis_uploads", per_axis_uploads},
    {"adjoint_lifetimes", adjoint_lifetimes},
    {"taped_kernels", taped_kernels},
};

}  // namespace

int main(int argc, char** argv) {
    const size_t before = rt::live.size();
    for (const Check& c : checks)
        if (argc > 1 && !strcmp(argv[1], c.name)) {
            c.run();
            CHECK(rt::live.size() == before && rt::streams.empty() && rt::graphs.empty());  // all given back
            std::printf("%s: %s (%d failures)\n", c.name, rt::failures ? "FAILED" : "ok", rt::failures);
            return rt::failures ? 1 : 0;
        }
    std::fprintf(stderr, "no such check\n");
    return 2;
}
