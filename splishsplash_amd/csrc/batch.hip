// batch.hip -- many independent DFSPH scenes stepped together
// (sph_dfsph_step_batch; no counterpart in the reference, which steps one
// scene: SimulatorBase::timeStep, SimulatorBase.cpp:959-1006).
//
// A step of every scene is cut at its two solves. The parts between them
// (neighbour search, boundary records, set-up sweeps, non-pressure forces,
// finalisation) run per scene on the scene's own stream, shared out over
// host threads. The solves -- nearly all of a step's launches -- run for all
// scenes at once: each Jacobi iteration is three launches in all (the
// acceleration sweep and the update over every scene's particles, one
// reduction block per scene), reading the scenes' states from a device
// table, and a scene whose solve has converged returns at entry. The
// iterations between two convergence checks are captured once as a HIP
// graph and replayed. Scenes are grouped by their lanes per particle, one
// batch per group.
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "dfsph.hpp"

namespace sph {
namespace {

// Host workers kept across the phases of a batch: run(n, f) calls f(k) for
// k < n over the workers and the calling thread, returns when all are done
// and rethrows the first error. Scene k's work goes to its own stream.
class Pool {
public:
    explicit Pool(size_t workers) {
        for (size_t t = 0; t < workers; t++) th_.emplace_back([this] { loop(); });
    }
    ~Pool() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            quit_ = true;
        }
        cv_.notify_all();
        for (auto &t : th_) t.join();
    }
    size_t size() const { return th_.size() + 1; }
    void run(size_t n, const std::function<void(size_t)> &f) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            job_ = &f;
            n_ = n;
            next_ = 0;
            busy_ = th_.size();
            failed_ = false;
            gen_++;
        }
        cv_.notify_all();
        work();
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [this] { return busy_ == 0; });
        job_ = nullptr;
        if (failed_) throw Error(code_, "batch: " + msg_);
    }

private:
    std::vector<std::thread> th_;
    std::mutex mu_;
    std::condition_variable cv_, done_;
    const std::function<void(size_t)> *job_ = nullptr;
    size_t n_ = 0, busy_ = 0;
    std::atomic<size_t> next_{0};
    unsigned long long gen_ = 0;
    bool quit_ = false, failed_ = false;
    int code_ = SPH_OK;
    std::string msg_;

    void work() {
        for (;;) {
            const size_t k = next_.fetch_add(1);
            if (k >= n_) return;
            try {
                (*job_)(k);
            } catch (const Error &e) {
                fail(e.code, e.what());
            } catch (const std::exception &e) {
                fail(SPH_ERR_INVALID, e.what());
            }
        }
    }
    void fail(int code, const std::string &m) {
        std::lock_guard<std::mutex> lk(mu_);
        if (!failed_) {
            failed_ = true;
            code_ = code;
            msg_ = m;
        }
        next_ = n_;  // the others stop taking scenes
    }
    void loop() {
        unsigned long long seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return quit_ || gen_ != seen; });
                if (quit_) return;
                seen = gen_;
            }
            work();
            {
                std::lock_guard<std::mutex> lk(mu_);
                busy_--;
            }
            done_.notify_all();
        }
    }
};

// The host form of xcd_block(): the particle block that hardware block b of
// a B-block launch works on (each XCD gets one contiguous range of blocks).
unsigned xcd_range(unsigned b, unsigned B) {
    const unsigned per = B / 8u, rem = B % 8u;
    const unsigned xcd = b % 8u, local = b / 8u;
    return xcd < rem ? xcd * (per + 1u) + local : rem * (per + 1u) + (xcd - rem) * per + local;
}

// Block map of a batched sweep over scenes of n[k] particles: entry q of the
// batched launch = (scene, particle block, partial-sum slot). The particle
// blocks of all scenes, concatenated, are spread over the XCDs as one
// launch's would be (contiguous ranges per XCD); the slot is the hardware
// block that takes the same particle block in the scene's own launch at these
// lanes, so the error partials, and with them every result, equal the scene's
// own. (A scene that takes 16 lanes alone and one in company has the same
// neighbour sums, but FP64 partials over 16 particles a block instead of 256:
// their totals, which decide when a solve ends and scale the CG's steps, may
// differ in the last bit.)
// With ids, entry k of n is scene ids[k] of the group's table (a map over
// a subset of the scenes).
std::vector<uint4> block_map(const std::vector<size_t> &n, int lanes, const std::vector<unsigned> *ids = nullptr) {
    std::vector<unsigned> first(n.size() + 1, 0);
    std::vector<std::vector<unsigned>> slot(n.size());
    for (size_t k = 0; k < n.size(); k++) {
        const unsigned nb = nblocks(n[k] * (size_t)lanes);
        first[k + 1] = first[k] + nb;
        slot[k].resize(nb);
        for (unsigned b = 0; b < nb; b++) slot[k][xcd_range(b, nb)] = b;
    }
    const unsigned NB = first.back();
    std::vector<uint4> m(NB);
    for (unsigned q = 0; q < NB; q++) {
        const unsigned r = xcd_range(q, NB);
        const size_t k = (size_t)(std::upper_bound(first.begin(), first.end(), r) - first.begin()) - 1;
        const unsigned lb = r - first[k];
        m[q] = make_uint4(ids ? (*ids)[k] : (unsigned)k, lb, slot[k][lb], 0u);
    }
    return m;
}

// One group of scenes with the same lanes per particle: the device table of
// their states, the block maps of the two sweeps, the convergence flags and
// the captured iteration chunks.
struct Group {
    std::vector<DFSPH *> scenes;
    int lanesA = 1, lanesJ = 1;
    DBuf<Dev> table;
    DBuf<uint4> mapA, mapJ;
    DBuf<int> done;
    unsigned nbA = 0, nbJ = 0;
    std::vector<size_t> sizes;  // particle counts the maps were built for
    std::map<int, hipGraphExec_t> graphs[2];  // [pressure][chunk]
    std::vector<Dev> hdev;
    std::vector<int> hdone;
    // maps over the scenes still iterating (rebuilt when some converge)
    DBuf<uint4> cmapA, cmapJ;
    unsigned cnbA = 0, cnbJ = 0;
    std::vector<uint4> hcA, hcJ;

    void compact(const std::vector<unsigned> &active, hipStream_t s) {
        std::vector<size_t> n;
        for (unsigned k : active) n.push_back(sizes[k]);
        hcA = block_map(n, lanesA, &active);
        hcJ = block_map(n, lanesJ, &active);
        cnbA = (unsigned)hcA.size();
        cnbJ = (unsigned)hcJ.size();
        cmapA.reserve(std::max<size_t>(nbA, 1));
        cmapJ.reserve(std::max<size_t>(nbJ, 1));
        if (cnbA) SPH_HIP(hipMemcpyAsync(cmapA.get(), hcA.data(), cnbA * sizeof(uint4), hipMemcpyHostToDevice, s));
        if (cnbJ) SPH_HIP(hipMemcpyAsync(cmapJ.get(), hcJ.data(), cnbJ * sizeof(uint4), hipMemcpyHostToDevice, s));
    }

    ~Group() { drop_graphs(); }
    void drop_graphs() {
        for (auto &g : graphs)
            for (auto &kv : g) (void)hipGraphExecDestroy(kv.second);
        graphs[0].clear();
        graphs[1].clear();
    }

    // (Re)builds the block maps when a particle count changed.
    void maps() {
        std::vector<size_t> now;
        for (DFSPH *s : scenes) now.push_back(s->n());
        if (now == sizes && nbA) return;
        for (DFSPH *s : scenes)
            SPH_REQUIRE(2 * (size_t)nblocks(s->n() * (size_t)lanesJ) <= s->partial_room(), SPH_ERR_STATE,
                        "batch: more error partials than the scene has room for");
        drop_graphs();
        sizes = now;
        const std::vector<uint4> a = block_map(now, lanesA), j = block_map(now, lanesJ);
        nbA = (unsigned)a.size();
        nbJ = (unsigned)j.size();
        mapA.reserve(std::max<size_t>(a.size(), 1));
        mapJ.reserve(std::max<size_t>(j.size(), 1));
        if (!a.empty()) SPH_HIP(hipMemcpy(mapA.get(), a.data(), a.size() * sizeof(uint4), hipMemcpyHostToDevice));
        if (!j.empty()) SPH_HIP(hipMemcpy(mapJ.get(), j.data(), j.size() * sizeof(uint4), hipMemcpyHostToDevice));
        table.reserve(scenes.size());
        done.reserve(scenes.size());
        hdev.resize(scenes.size());
        hdone.resize(scenes.size());
    }
};

}  // namespace

struct BatchRunner {
    hipStream_t stream = nullptr;
    std::vector<std::unique_ptr<Group>> groups;
    std::vector<hipEvent_t> ev;  // per scene: its part of the step is enqueued
    hipEvent_t solved = nullptr;
    std::vector<unsigned long long> ids;
    bool graphs = true;
    size_t threads = 16;
    std::unique_ptr<Pool> pool;

    void parallel_scenes(size_t n, const std::function<void(size_t)> &f) {
        if (!pool || pool->size() != std::max<size_t>(1, threads)) pool.reset(new Pool(std::max<size_t>(1, threads) - 1));
        pool->run(n, f);
    }

    ~BatchRunner() {
        groups.clear();
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        if (solved) (void)hipEventDestroy(solved);
        if (stream) (void)hipStreamDestroy(stream);
    }

    // The batch stream and the per-scene events (before a step's first part).
    void resources(size_t n) {
        if (!stream) SPH_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        if (!solved) SPH_HIP(hipEventCreateWithFlags(&solved, hipEventDisableTiming));
        while (ev.size() < n) {
            hipEvent_t e;
            SPH_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            ev.push_back(e);
        }
    }

    // Groups and block maps (once each scene's lanes are known).
    void setup(const std::vector<DFSPH *> &all) {
        // group by the scenes' lanes: the same scenes at other lanes (a scene
        // that has grown, or is stepped in other company) are another group
        std::map<std::pair<int, int>, std::vector<DFSPH *>> by;
        for (DFSPH *s : all) by[{s->lanes_accel(), s->lanes_jacobi()}].push_back(s);
        bool same = by.size() == groups.size();
        if (same) {
            size_t g = 0;
            for (auto &kv : by) {
                const Group &h = *groups[g++];
                same = same && h.scenes == kv.second && h.lanesA == kv.first.first && h.lanesJ == kv.first.second;
            }
        }
        if (!same) {
            groups.clear();
            for (auto &kv : by) {
                auto g = std::make_unique<Group>();
                g->scenes = kv.second;
                g->lanesA = kv.first.first;
                g->lanesJ = kv.first.second;
                groups.push_back(std::move(g));
            }
        }
        for (auto &g : groups) g->maps();
    }

    // The solve of every scene (the scenes' parts before it are enqueued on
    // their streams and marked by ev[k]).
    void solve(const std::vector<DFSPH *> &all, bool pressure, std::vector<int> &iterations) {
        for (size_t k = 0; k < all.size(); k++) SPH_HIP(hipStreamWaitEvent(stream, ev[k], 0));
        for (auto &gp : groups) {
            Group &g = *gp;
            const unsigned ns = (unsigned)g.scenes.size();
            int maxIt = 1;
            std::vector<int> pred(ns);
            for (size_t k = 0; k < ns; k++) {
                g.hdev[k] = g.scenes[k]->device_state();
                pred[k] = g.scenes[k]->first_chunk(pressure);
                maxIt = std::max(maxIt, pressure ? g.scenes[k]->P.max_iterations : g.scenes[k]->P.max_iterations_v);
            }
            // the first chunk runs to the median predicted count; the scenes
            // that then still iterate go on in a compacted launch
            std::nth_element(pred.begin(), pred.begin() + ns / 2, pred.end());
            int chunk = std::max(1, pred[ns / 2]);
            SPH_HIP(hipMemcpyAsync(g.table.get(), g.hdev.data(), ns * sizeof(Dev), hipMemcpyHostToDevice, stream));
            int launched = 0;
            std::vector<unsigned> active(ns);
            for (unsigned k = 0; k < ns; k++) active[k] = k;
            bool compacted = false;
            for (;;) {
                const int c = std::min(chunk, maxIt - launched);
                if (compacted) {
                    // only the scenes still iterating (a converged scene's
                    // blocks would return at entry, but still be dispatched)
                    for (int i = 0; i < c; i++)
                        launch_batch_iteration(pressure, g.lanesA, g.lanesJ, g.table.get(), g.cmapA.get(), g.cnbA,
                                               g.cmapJ.get(), g.cnbJ, ns, stream);
                } else {
                    run_chunk(g, pressure, c);
                }
                launched += c;
                launch_batch_done(pressure, g.table.get(), ns, g.done.get(), stream);
                SPH_HIP(hipMemcpyAsync(g.hdone.data(), g.done.get(), ns * sizeof(int), hipMemcpyDeviceToHost, stream));
                SPH_HIP(hipStreamSynchronize(stream));
                std::vector<unsigned> still;
                for (unsigned k : active)
                    if (g.hdone[k] == 0) still.push_back(k);
                if (still.empty() || launched >= maxIt) break;
                if (still.size() < active.size()) {
                    active.swap(still);
                    g.compact(active, stream);
                    compacted = true;
                }
                chunk = 2;  // past the predicted count: two iterations per round trip
            }
        }
        SPH_HIP(hipEventRecord(solved, stream));
        parallel_scenes(all.size(), [&](size_t k) {
            SPH_HIP(hipStreamWaitEvent(all[k]->stream, solved, 0));
            iterations[k] = all[k]->solve_result(pressure);
        });
    }

    // c iterations of the group: replayed from a captured graph.
    void run_chunk(Group &g, bool pressure, int c) {
        const unsigned ns = (unsigned)g.scenes.size();
        if (!graphs) {
            for (int i = 0; i < c; i++)
                launch_batch_iteration(pressure, g.lanesA, g.lanesJ, g.table.get(), g.mapA.get(), g.nbA, g.mapJ.get(),
                                       g.nbJ, ns, stream);
            return;
        }
        auto &cache = g.graphs[pressure ? 1 : 0];
        auto it = cache.find(c);
        if (it == cache.end()) {
            hipGraph_t graph;
            SPH_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
            for (int i = 0; i < c; i++)
                launch_batch_iteration(pressure, g.lanesA, g.lanesJ, g.table.get(), g.mapA.get(), g.nbA, g.mapJ.get(),
                                       g.nbJ, ns, stream);
            SPH_HIP(hipStreamEndCapture(stream, &graph));
            hipGraphExec_t exec;
            const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            SPH_HIP(e);
            it = cache.emplace(c, exec).first;
        }
        SPH_HIP(hipGraphLaunch(it->second, stream));
    }

    void step(const std::vector<DFSPH *> &all) {
        resources(all.size());
        std::vector<char> div(all.size(), 0);
        std::vector<int> its(all.size(), 0);
        parallel_scenes(all.size(), [&](size_t k) {
            div[k] = all[k]->step_begin() ? 1 : 0;
            SPH_HIP(hipEventRecord(ev[k], all[k]->stream));
        });
        setup(all);  // a search may have changed a scene's lanes
        bool anydiv = false;
        for (char d : div) anydiv = anydiv || d;
        if (anydiv) {
            // a scene without the divergence solver reads as converged at once
            solve(all, false, its);
        }
        parallel_scenes(all.size(), [&](size_t k) {
            if (div[k]) all[k]->step_after_divergence(its[k]);
            all[k]->step_middle(div[k] != 0);
            SPH_HIP(hipEventRecord(ev[k], all[k]->stream));
        });
        solve(all, true, its);
        parallel_scenes(all.size(), [&](size_t k) { all[k]->step_after_pressure(its[k]); });
    }
};

// The runner of the last batch (its stream, tables and graphs are kept for
// the next call on the same scenes).
static std::mutex g_batch_mu;
static std::unique_ptr<BatchRunner> g_batch;

void step_batched(const std::vector<DFSPH *> &all, int n_steps, size_t threads, bool graphs) {
    std::lock_guard<std::mutex> lk(g_batch_mu);
    std::vector<unsigned long long> ids;
    for (DFSPH *s : all) ids.push_back(s->serial());
    if (!g_batch || g_batch->ids != ids) {
        g_batch.reset(new BatchRunner());
        g_batch->ids = ids;
    }
    g_batch->threads = threads;
    if (g_batch->graphs != graphs) {
        for (auto &g : g_batch->groups) g->drop_graphs();
        g_batch->graphs = graphs;
    }
    for (int st = 0; st < n_steps; st++) g_batch->step(all);
    g_batch->parallel_scenes(all.size(), [&](size_t k) { all[k]->sync(); });
}

}  // namespace sph
