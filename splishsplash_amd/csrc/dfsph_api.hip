// dfsph_api.hip -- sph_dfsph_* : C-ABI over the device-resident DFSPH step
// (TimeStepDFSPH and the state it steps; see include/sph_capi.h).
#include <algorithm>
#include <chrono>
#include <atomic>
#include <cstring>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "dfsph.hpp"

using namespace sph;

struct sph_dfsph {
    std::unique_ptr<DFSPH> s;
};

#define DCHK(h) SPH_REQUIRE((h) != nullptr && (h)->s, SPH_ERR_INVALID, "null handle")

extern "C" {

void sph_dfsph_default_params(sph_dfsph_params_t *p) {
    if (!p) return;
    std::memset(p, 0, sizeof(*p));
    p->particle_radius = 0.025;
    p->density0 = 1000.0;
    p->gravity[1] = -9.81;
    p->time_step_size = 0.001;
    p->cfl_method = 1;
    p->cfl_factor = 0.5;
    p->cfl_min_time_step_size = 0.0001;
    p->cfl_max_time_step_size = 0.005;
    p->min_iterations = 2;
    p->max_iterations = 100;
    p->max_error = 0.01;
    p->max_iterations_v = 100;
    p->max_error_v = 0.1;
    p->enable_divergence_solver = 1;
    p->viscosity_method = SPH_VISCOSITY_NONE;
    p->viscosity = 0.01;
    p->visco_max_iter = 100;
    p->visco_max_error = 0.01;
    p->boundary_handling_method = SPH_BOUNDARY_BENDER2019;
}

int sph_dfsph_create(const sph_dfsph_params_t *params, sph_dfsph_t *out) {
    return guarded([&] {
        SPH_REQUIRE(params && out, SPH_ERR_INVALID, "null argument");
        auto *h = new sph_dfsph();
        try {
            h->s.reset(new DFSPH(*params));
        } catch (...) {
            delete h;
            throw;
        }
        *out = h;
    });
}

int sph_dfsph_destroy(sph_dfsph_t s) {
    return guarded([&] { delete s; });
}

int sph_dfsph_set_fluid(sph_dfsph_t s, const float *x, const float *v, size_t n) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(x && n > 0, SPH_ERR_INVALID, "need at least one particle");
        s->s->set_fluid(x, v, n);
    });
}

int sph_dfsph_add_boundary_particles(sph_dfsph_t s, const float *x, size_t n) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(x || n == 0, SPH_ERR_INVALID, "null positions");
        s->s->add_boundary(x, n);
    });
}

int sph_dfsph_set_volume_map_box(sph_dfsph_t s, const double box_min[3], const double box_max[3], int invert,
                                 double thickness, const unsigned resolution[3]) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(box_min && box_max && resolution, SPH_ERR_INVALID, "null argument");
        s->s->set_volume_map_box(box_min, box_max, invert, thickness, resolution);
    });
}

int sph_dfsph_add_volume_map_sphere(sph_dfsph_t s, const double centre[3], double radius, int invert,
                                    double thickness, const unsigned resolution[3]) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(centre && resolution, SPH_ERR_INVALID, "null argument");
        SPH_REQUIRE(radius > 0, SPH_ERR_INVALID, "radius must be > 0");
        Shape sh;
        sh.kind = SHAPE_SPHERE;
        for (int c = 0; c < 3; c++) sh.centre[c] = centre[c];
        sh.radius = radius;
        sh.invert = invert;
        sh.thickness = thickness;
        s->s->add_volume_map(sh, resolution);
    });
}

int sph_dfsph_add_volume_map_mesh(sph_dfsph_t s, const double *vertices, size_t n_vertices, const unsigned *faces,
                                  size_t n_faces, int invert, double thickness, const unsigned resolution[3]) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(resolution, SPH_ERR_INVALID, "null resolution");
        s->s->add_volume_map_mesh(vertices, n_vertices, faces, n_faces, invert, thickness, resolution);
    });
}

int sph_dfsph_init(sph_dfsph_t s) {
    return guarded([&] {
        DCHK(s);
        s->s->init();
    });
}

int sph_dfsph_reset(sph_dfsph_t s) {
    return guarded([&] {
        DCHK(s);
        s->s->reset();
    });
}

int sph_dfsph_emit_particles(sph_dfsph_t s, const float *x, const float *v, size_t n) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(x || n == 0, SPH_ERR_INVALID, "null positions");
        s->s->emit_particles(x, v, n);
    });
}

int sph_dfsph_set_simulation_method(sph_dfsph_t s, int method) {
    return guarded([&] {
        DCHK(s);
        s->s->set_method(method);
    });
}

int sph_dfsph_set_wcsph(sph_dfsph_t s, double stiffness, double exponent) {
    return guarded([&] {
        DCHK(s);
        s->s->set_wcsph(stiffness, exponent);
    });
}

int sph_dfsph_add_emitter(sph_dfsph_t s, const sph_emitter_t *e) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(e != nullptr, SPH_ERR_INVALID, "null emitter");
        sph::EmitterDesc d;
        d.type = e->type;
        d.width = e->width;
        d.height = e->height;
        for (int c = 0; c < 3; c++) d.x[c] = e->translation[c];
        for (int c = 0; c < 9; c++) d.R[c] = e->rotation[c];
        d.velocity = e->velocity;
        d.start = e->emit_start_time;
        d.end = e->emit_end_time;
        s->s->add_emitter(d);
    });
}

int sph_dfsph_set_emitter_reuse(sph_dfsph_t s, int enable, const double box_min[3], const double box_max[3]) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(!enable || (box_min && box_max), SPH_ERR_INVALID, "null reuse box");
        s->s->set_emitter_reuse(enable != 0, box_min, box_max);
    });
}

int sph_dfsph_set_max_emitter_particles(sph_dfsph_t s, size_t max_particles) {
    return guarded([&] {
        DCHK(s);
        s->s->set_max_emitter_particles(max_particles);
    });
}

int sph_dfsph_emitter_counts(sph_dfsph_t s, size_t *emitted, size_t *reused) {
    return guarded([&] {
        DCHK(s);
        if (emitted) *emitted = s->s->emitted();
        if (reused) *reused = s->s->reused();
    });
}

int sph_dfsph_set_body_motion(sph_dfsph_t s, unsigned obj, const double position[3], const double rotation[9],
                              const double velocity[3], const double angular_velocity[3], int kind) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(position && rotation && velocity && angular_velocity, SPH_ERR_INVALID,
                    "sph_dfsph_set_body_motion: null argument");
        s->s->set_body_motion(obj, position, rotation, velocity, angular_velocity, kind);
    });
}

int sph_dfsph_get_body_force(sph_dfsph_t s, unsigned obj, double force[3], double torque[3], int clear) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(force && torque, SPH_ERR_INVALID, "sph_dfsph_get_body_force: null argument");
        s->s->body_force(obj, force, torque, clear != 0);
    });
}

int sph_dfsph_set_fluid_models(sph_dfsph_t s, const unsigned *model, size_t n, const double *materials,
                               unsigned n_models) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE((model || n == 0) && materials, SPH_ERR_INVALID, "sph_dfsph_set_fluid_models: null argument");
        s->s->set_fluid_models(model, n, materials, n_models);
    });
}

int sph_dfsph_get_body_reference(sph_dfsph_t s, unsigned obj, double position[3], double *max_dist) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(position && max_dist, SPH_ERR_INVALID, "sph_dfsph_get_body_reference: null argument");
        s->s->body_reference(obj, position, max_dist);
    });
}

int sph_dfsph_step(sph_dfsph_t s, int n_steps) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(n_steps >= 0, SPH_ERR_INVALID, "n_steps must be >= 0");
        for (int i = 0; i < n_steps; i++) s->s->step();
        s->s->sync();
    });
}

// How sph_dfsph_step_batch runs (sph_dfsph_set_batch_mode).
static std::atomic<int> g_batch_mode{3};

int sph_dfsph_set_batch_mode(int mode) {
    return guarded([&] {
        SPH_REQUIRE(mode >= 0 && mode <= 3, SPH_ERR_INVALID, "batch mode must be 0, 1, 2 or 3");
        g_batch_mode = mode;
    });
}

namespace {

// n_steps of every scene, scene by scene: the handles are shared out over T
// host threads by particle count (longest processing time first) and each
// thread interleaves its scenes step by step.
void step_threads(sph_dfsph_t *handles, size_t n, int n_steps, size_t T) {
    std::vector<size_t> order(n);
    for (size_t k = 0; k < n; k++) order[k] = k;
    std::sort(order.begin(), order.end(), [&](size_t a, size_t b) { return handles[a]->s->n() > handles[b]->s->n(); });
    std::vector<std::vector<size_t>> work(T);
    std::vector<size_t> load(T, 0);
    for (size_t k : order) {
        const size_t t = (size_t)(std::min_element(load.begin(), load.end()) - load.begin());
        work[t].push_back(k);
        load[t] += std::max<size_t>(handles[k]->s->n(), 1);
    }
    std::atomic<bool> failed{false};
    std::mutex mu;
    int code = SPH_OK;
    std::string msg;
    auto run = [&](size_t t) {
        try {
            for (int st = 0; st < n_steps && !failed.load(); st++)
                for (size_t k : work[t]) handles[k]->s->step();
            for (size_t k : work[t]) handles[k]->s->sync();
        } catch (const Error &e) {
            std::lock_guard<std::mutex> lk(mu);
            if (!failed.exchange(true)) code = e.code, msg = e.what();
        } catch (const std::exception &e) {
            std::lock_guard<std::mutex> lk(mu);
            if (!failed.exchange(true)) code = SPH_ERR_INVALID, msg = e.what();
        }
    };
    std::vector<std::thread> pool;
    for (size_t t = 1; t < T; t++) pool.emplace_back(run, t);
    run(0);
    for (auto &th : pool) th.join();
    if (failed) throw Error(code, "batch: " + msg);
}

// Mode 3: the first steps of a set of scenes alternate between scene by
// scene on host threads and batched solves from graphs, one step timed per
// way after one untimed (set-up, graph capture); the faster way
// runs from then on. A different set of handles is timed again.
struct AutoChoice {
    std::vector<unsigned long long> ids;
    int probe = 0;        // steps of the trial so far (4 in all)
    double t[2] = {0, 0}; // seconds of the timed step: threads, graphs
    int choice = -1;      // 0 threads, 2 graphs
};
std::mutex g_auto_mu;
AutoChoice g_auto;

}  // namespace

int sph_dfsph_step_batch(sph_dfsph_t *handles, size_t n, int n_steps, int threads) {
    return guarded([&] {
        SPH_REQUIRE(handles || n == 0, SPH_ERR_INVALID, "null handle array");
        SPH_REQUIRE(n_steps >= 0, SPH_ERR_INVALID, "n_steps must be >= 0");
        SPH_REQUIRE(threads >= 0, SPH_ERR_INVALID, "threads must be >= 0");
        if (n == 0 || n_steps == 0) return;
        std::set<sph_dfsph_t> seen;
        for (size_t k = 0; k < n; k++) {
            DCHK(handles[k]);
            SPH_REQUIRE(seen.insert(handles[k]).second, SPH_ERR_INVALID, "a handle appears twice in the batch");
        }
        struct Company {  // tells every scene how many particles step together
            sph_dfsph_t *h;
            size_t n;
            Company(sph_dfsph_t *hh, size_t nn) : h(hh), n(nn) {
                size_t total = 0;
                for (size_t k = 0; k < n; k++) total += h[k]->s->n();
                for (size_t k = 0; k < n; k++) h[k]->s->set_company(total);
            }
            ~Company() {
                for (size_t k = 0; k < n; k++) h[k]->s->set_company(0);
            }
        } company(handles, n);
        // A first step sets a handle up (boundary maps, buffers, list room)
        // and picks its lanes per particle, by which batched solves group the
        // scenes: it runs here for every handle, one handle at a time, before
        // host threads or batched solves take over. (A run whose fresh
        // handles took first steps concurrently has faulted, cause not found.)
        bool pending = false;
        for (size_t k = 0; k < n; k++) pending = pending || handles[k]->s->first_step_pending();
        if (pending) {
            for (size_t k = 0; k < n; k++) handles[k]->s->step();
            for (size_t k = 0; k < n; k++) handles[k]->s->sync();
            if (--n_steps == 0) return;
        }
        const size_t T = std::min<size_t>(n, threads > 0 ? (size_t)threads : 16);
        bool ok = true;
        for (size_t k = 0; k < n; k++)
            ok = ok && handles[k]->s->batchable() &&
                 handles[k]->s->P.enable_divergence_solver == handles[0]->s->P.enable_divergence_solver;
        std::vector<DFSPH *> all;
        for (size_t k = 0; k < n; k++) all.push_back(handles[k]->s.get());
        const int mode = g_batch_mode;
        if (!ok || mode == 0) {
            step_threads(handles, n, n_steps, T);
            return;
        }
        if (mode != 3) {
            step_batched(all, n_steps, T, mode == 2);
            return;
        }
        std::lock_guard<std::mutex> lk(g_auto_mu);
        std::vector<unsigned long long> ids;
        for (DFSPH *s : all) ids.push_back(s->serial());
        if (g_auto.ids != ids) {
            g_auto = AutoChoice{};
            g_auto.ids = ids;
        }
        int left = n_steps;
        while (left > 0 && g_auto.choice < 0) {
            const int way = g_auto.probe < 2 ? 0 : 2;
            const auto t0 = std::chrono::steady_clock::now();
            if (way == 0)
                step_threads(handles, n, 1, T);
            else
                step_batched(all, 1, T, true);
            const double dt = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            if (g_auto.probe % 2 == 1) g_auto.t[way == 0 ? 0 : 1] = dt;
            left--;
            if (++g_auto.probe == 4) g_auto.choice = g_auto.t[0] <= g_auto.t[1] ? 0 : 2;
        }
        if (left == 0) return;
        if (g_auto.choice == 0)
            step_threads(handles, n, left, T);
        else
            step_batched(all, left, T, true);
    });
}

// The way mode 3 chose for the last set of scenes (-1: still timing).
int sph_dfsph_batch_choice(void) {
    std::lock_guard<std::mutex> lk(g_auto_mu);
    return g_auto.choice;
}

int sph_dfsph_stage(sph_dfsph_t s, int stage) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(stage >= 0 && stage < SPH_STAGE_COUNT, SPH_ERR_INVALID, "unknown stage");
        s->s->stage(stage);
    });
}

int sph_dfsph_num_particles(sph_dfsph_t s, size_t *out) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(out, SPH_ERR_INVALID, "null argument");
        *out = s->s->n();
    });
}

int sph_dfsph_get_field(sph_dfsph_t s, const char *name, void *host, size_t bytes) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(name && host, SPH_ERR_INVALID, "null argument");
        s->s->get_field(name, host, bytes);
    });
}

int sph_dfsph_set_field(sph_dfsph_t s, const char *name, const void *host, size_t bytes) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(name && host, SPH_ERR_INVALID, "null argument");
        s->s->set_field(name, host, bytes);
    });
}

int sph_dfsph_get_neighbors(sph_dfsph_t s, int boundary, unsigned *offsets, unsigned *indices, size_t capacity,
                            size_t *nnz) {
    return guarded([&] {
        DCHK(s);
        s->s->get_neighbors(boundary, offsets, indices, capacity, nnz);
    });
}

int sph_dfsph_set_warm_start_model(sph_dfsph_t s, int solver, const float *theta) {
    return guarded([&] {
        DCHK(s);
        s->s->set_warm_start_model(solver, theta);
    });
}

int sph_dfsph_set_warm_start_mode(sph_dfsph_t s, int solver, int mode) {
    return guarded([&] {
        DCHK(s);
        s->s->set_warm_start_mode(solver, mode);
    });
}

int sph_dfsph_set_warm_start_policy(sph_dfsph_t s, int solver, int min_prev_iterations) {
    return guarded([&] {
        DCHK(s);
        s->s->set_warm_start_policy(solver, min_prev_iterations);
    });
}

int sph_dfsph_collect_training(sph_dfsph_t s, int solver, unsigned stride, size_t capacity) {
    return guarded([&] {
        DCHK(s);
        s->s->collect_training(solver, stride, capacity);
    });
}

int sph_dfsph_get_training(sph_dfsph_t s, int solver, float *x, float *t, size_t capacity, size_t *n) {
    return guarded([&] {
        DCHK(s);
        s->s->get_training(solver, x, t, capacity, n);
    });
}

int sph_dfsph_get_counters(sph_dfsph_t s, sph_dfsph_counters_t *out) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(out, SPH_ERR_INVALID, "null argument");
        s->s->counters(out);
    });
}

int sph_dfsph_set_time(sph_dfsph_t s, double time, double time_step_size) {
    return guarded([&] {
        DCHK(s);
        s->s->set_time(time, time_step_size);
    });
}

int sph_dfsph_write_particles(sph_dfsph_t s, const char *path, const char *fields) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(path, SPH_ERR_INVALID, "null path");
        write_particles(*s->s, path, fields);
    });
}

int sph_dfsph_save_state(sph_dfsph_t s, const char *prefix) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(prefix, SPH_ERR_INVALID, "null path");
        const std::string pre(prefix);
        write_state(*s->s, pre + "_particle_Fluid.bgeo");
        sph_dfsph_counters_t c;
        s->s->counters(&c);
        // time, step size and the emitter system's progress
        // (EmitterSystem::saveState, EmitterSystem.cpp:120-126)
        FILE *f = std::fopen((pre + ".json").c_str(), "w");
        SPH_REQUIRE(f, SPH_ERR_INVALID, "cannot write " + pre + ".json");
        std::fprintf(f, "{\"time\": %.17g, \"timeStepSize\": %.17g, \"numParticles\": %zu, \"emitted\": %zu, "
                        "\"reused\": %zu, \"emitters\": [",
                     c.time, c.time_step_size, s->s->n(), s->s->emitted(), s->s->reused());
        const auto &em = s->s->emitters();
        for (size_t k = 0; k < em.size(); k++)
            std::fprintf(f, "%s[%.17g, %u]", k ? ", " : "", em[k].next, em[k].counter);
        std::fprintf(f, "]}\n");
        SPH_REQUIRE(std::fclose(f) == 0, SPH_ERR_INVALID, "write failed: " + pre + ".json");
    });
}

int sph_dfsph_load_state(sph_dfsph_t s, const char *prefix) {
    return guarded([&] {
        DCHK(s);
        SPH_REQUIRE(prefix, SPH_ERR_INVALID, "null path");
        const std::string pre(prefix);
        FILE *f = std::fopen((pre + ".json").c_str(), "r");
        SPH_REQUIRE(f, SPH_ERR_INVALID, "cannot open " + pre + ".json");
        double t = 0.0, h = 0.0;
        size_t n = 0, emitted = 0, reused = 0;
        int got = std::fscanf(f, " {\"time\": %lf, \"timeStepSize\": %lf, \"numParticles\": %zu", &t, &h, &n);
        std::vector<std::pair<double, unsigned>> prog;
        bool has_emit = false;
        if (got == 3 && std::fscanf(f, " , \"emitted\": %zu , \"reused\": %zu , \"emitters\": [", &emitted,
                                    &reused) == 2) {
            has_emit = true;
            double next;
            unsigned counter;
            while (std::fscanf(f, " [ %lf , %u ]", &next, &counter) == 2) {
                prog.emplace_back(next, counter);
                if (std::fscanf(f, " ,") == EOF) break;
            }
        }
        std::fclose(f);
        SPH_REQUIRE(got == 3, SPH_ERR_INVALID, "malformed " + pre + ".json");
        SPH_REQUIRE(n >= s->s->n(), SPH_ERR_INVALID,
                    "the state holds " + std::to_string(n) + " particles, fewer than the handle's " +
                        std::to_string(s->s->n()));
        SPH_REQUIRE(!has_emit || prog.size() == s->s->emitters().size(), SPH_ERR_INVALID,
                    "the state holds " + std::to_string(prog.size()) + " emitters, the handle " +
                        std::to_string(s->s->emitters().size()));
        if (n == 0) return;
        s->s->init_if_needed();
        read_state(*s->s, pre + "_particle_Fluid.bgeo");
        s->s->set_time(t, h);
        if (has_emit) {
            for (size_t k = 0; k < prog.size(); k++) s->s->set_emitter_progress(k, prog[k].first, prog[k].second);
            s->s->set_emit_counts(emitted, reused);
        }
    });
}

int sph_dfsph_enable_timing(sph_dfsph_t s, int enable) {
    return guarded([&] {
        DCHK(s);
        s->s->timer.enabled = enable != 0;
    });
}

int sph_dfsph_time_only(sph_dfsph_t s, const char *names) {
    return guarded([&] {
        DCHK(s);
        auto &only = s->s->timer.only;
        only.clear();
        if (!names) return;
        std::string cur;
        for (const char *c = names;; c++) {
            if (*c == ',' || *c == 0) {
                if (!cur.empty()) only.push_back(cur);
                cur.clear();
                if (*c == 0) break;
            } else {
                cur.push_back(*c);
            }
        }
    });
}

int sph_dfsph_set_lanes_per_particle(sph_dfsph_t s, int lanes) {
    return guarded([&] {
        DCHK(s);
        s->s->set_lanes_per_particle(lanes);
    });
}

int sph_dfsph_kernel_stats(sph_dfsph_t s, int k, const char **name, long long *launches, double *total_ms,
                           int *count) {
    return guarded([&] {
        DCHK(s);
        s->s->sync();
        s->s->timer.collect();
        auto &st = s->s->timer.stats;
        if (count) *count = (int)st.size();
        if (k < 0 || k >= (int)st.size()) return;
        if (name) *name = st[k].name.c_str();
        if (launches) *launches = st[k].launches;
        if (total_ms) *total_ms = st[k].ms;
    });
}

int sph_dfsph_reset_kernel_stats(sph_dfsph_t s) {
    return guarded([&] {
        DCHK(s);
        s->s->sync();
        s->s->timer.reset();
    });
}

int sph_dfsph_synchronize(sph_dfsph_t s) {
    return guarded([&] {
        DCHK(s);
        s->s->sync();
    });
}

}  // extern "C"
