// dfsph.hpp -- device-resident DFSPH time step (TimeStepDFSPH,
// SPlisHSPlasH/DFSPH/TimeStepDFSPH.cpp) with its neighbour search, Akinci2012
// and Bender2019 boundaries, XSPH and the Weiler2018 implicit viscosity.
#pragma once
#include <array>
#include <memory>
#include <string>
#include <vector>

#include "common.hpp"
#include "grid.hpp"
#include "kernel_math.hpp"
#include "volume_map.hpp"

namespace sph {

// Scalars shared by host and kernels, resident in device memory so that
// time-step control and solver convergence never need a host round trip
// inside a step.
struct Ctl {
    double h;          // TimeManager time step size
    double h_step;     // h cached at the start of the step (TimeStepDFSPH.cpp:121)
    double time;
    double avg_err;    // last pressure iteration, average density error
    double avg_err_v;  // last divergence iteration
    double avg_over, avg_over_v;  // excess (positive residual where p > 0), same units
    double cg_rhs2, cg_thresh, cg_absNew, cg_alpha, cg_beta, cg_r2;
    int it, done;      // pressure solver
    int it_v, done_v;  // divergence solver
    int cg_it, cg_done;
    int it_prev;       // pressure iterations of the previous solve (CFL method 2)
    int chk_acc, chk_acc_v;  // several fluid models: every model so far met its tolerance
    int flags;         // bit0: non-finite value in a reduction
    unsigned maxcnt_f, maxcnt_b;
    unsigned ovf16;               // a packed list difference did not fit
    unsigned tiles_over;          // tiles that keep no slots (see k_tile_lists)
    double kref, kref_v;          // stiffness scales of the learned start
    unsigned nlearn, nlearn_v;    // particles that kept the learned start
    unsigned nsamp, nsamp_v;      // training samples written
    double t_prev;                // time at the start of the last completed step
};

// Everything a sweep kernel needs, passed by value.
struct Dev {
    unsigned n, stride;
    float4 *x, *v, *v2, *a, *ap, *vdiff, *xc, *vmb;
    const unsigned *state;  // ParticleState per particle (0 active); null: all active
    float *rho, *alpha, *radv, *p, *pv;
    const unsigned *nf, *cf, *nb, *cb;
    // Packed fluid lists (null when a slot difference does not fit 16 bits):
    // neighbours 2w and 2w + 1 of particle i as int16 differences j - i in
    // the low and high halves of nf16[w * stride + i]. The solver sweeps read
    // these -- half the index bytes and index loads of nf.
    const unsigned *nf16;
    // Tiled lists (null where nf16 is and unless they pay): the union
    // of the neighbours of particles b TILE .. b TILE + TILE - 1, tcount[b]
    // slots (0: more than TILE_CAP, or too far apart), as int16 differences
    // slot - b TILE, two per word, at tslot[b TILE_CAP / 2]; and the lists
    // of those particles as 16-bit places in the union, the words of nf16 by
    // quads: words 4g, 4g + 2, 4g + 1, 4g + 3 of particle i at
    // nt16[4 (g stride + i)], g < quads16. One or two lanes of the particle
    // then each load their share of a quad at once.
    const unsigned *nt16, *tslot, *tcount;
    unsigned quads16;
    const float4 *bx;  // Akinci particles (x, y, z, volume), cell-sorted
    int bmode;         // 0 none, 1 Akinci2012, 2 Bender2019, 3 Koschier2017
    unsigned nvm;      // map slots: vmb[o * stride + i], entries with
                       // w > 0 first (object order), then w = 0; w is V_b
                       // (Bender2019) or rho_b (Koschier2017)
    float4 *dmg;       // Koschier2017: grad rho_b per slot, same layout
    // Moving volume maps (animated or dynamic bodies); all null or 0 while
    // every body is at rest. vmv[o * stride + i] = (velocity of the body at
    // the boundary point of slot o, object index), packed like vmb.
    const float4 *vmv;
    const float4 *body;  // body[o] = (omega, dynamic ? 1 : 0), body[nbody + o] = (reference point, 0)
    unsigned nbody;
    double bodyMaxVel;   // largest |vel + omega x (maxDist, 0, 0)| of the moving bodies (CFL)
    double *bpart;       // per-block force and torque partials: [block][body][6]
    double *bforce;      // accumulated force and torque per body: [body][6]
    // Several fluid models (null `model`: one model with the scalars above).
    // model[i] is particle i's model; the solver sweeps of a model take its
    // particles only (solveModel, -1: every particle). Per model: rest
    // density, mass, viscosity d nu and d nu_b, XSPH coefficients, count.
    const unsigned *model;
    int solveModel;
    unsigned nmodel;
    float rho0m[8], massm[8], svm[8], svbm[8], xsm[8], xsbm[8];
    unsigned countm[8];
    float sphereVol;   // 4/3 pi h^3 (Koschier2017 viscosity samples)
    float V, rho0, eps, mass;
    float3 grav;
    KernelConst K;
    Ctl *ctl;
    double *partial;
    // solver parameters
    int minIt, maxIt, maxItV;
    double maxError, maxErrorV;
    float xsph, xsphB;
    float svisc, sviscB;  // Viscosity_Standard: d nu, d nu_b (0: off)
    int cflMethod;
    double cflFactor, cflMin, cflMax, radius;
    // Weiler2018
    float4 *minv;  // 2 float4 per particle: symmetric 3x3 inverse (xx xy xz yy | yz zz - -)
    float4 *cgx, *cgr, *cgp, *cgz, *cgt;
    float mu, mub, hs2;
    int viscoMaxIt;
    double viscoTol;
    // learned warm start
    int strictP, strictV;    // solves started from the network: also bound the excess
    float *feats, *feats_v;  // 8 floats per particle
    float *pred, *kprev;     // network output, previous-step stiffness
    float4 *ap2;             // pressure accelerations of the predicted start
    float *sx, *st, *sx_v, *st_v;
    unsigned scap, scap_v, sstride, sstride_v, soff;
};

// One emitter (Emitter.h:14-70): a width x height grid (type 0) or a disc
// of width particles across (type 1) leaving `x` along column 0 of the
// row-major rotation R, at `velocity`, between the start and end times.
struct EmitterDesc {
    int type = 0;
    unsigned width = 0, height = 0;
    double x[3] = {0, 0, 0};
    double R[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    double velocity = 0, start = 0, end = 0;
    double next = 0;       // m_nextEmitTime
    unsigned counter = 0;  // m_emitCounter
};

// Particles per tile of the tiled lists, and the slots a tile may gather (see
// k_tile_lists): a tile along a row of cells of fluid at rest has 1,300 to
// 1,500, at most 1,930 in a collapsing column. 24 bytes a slot let three
// blocks of k_jacobi_tile share a CU, 16 five of k_accel_tile.
constexpr unsigned TILE = 256, TILE_CAP = 1856;

// Below this many particles the lanes per particle only weigh time (see
// small_lanes), from it on they fix the order of the sums (see
// DFSPH::pick_lanes).
constexpr size_t SMALL_PARTICLES = 65536;

class DFSPH;
// Steps the scenes n_steps times together (batch.hip): their solves run as
// batched launches (replayed from captured HIP graphs when `graphs`), the
// rest of each step per scene on up to `threads` host threads. Every scene
// must be batchable() with the same divergence-solver setting.
void step_batched(const std::vector<DFSPH *> &scenes, int n_steps, size_t threads, bool graphs);

// One Jacobi iteration (accelerations, update, error reduction) of many
// scenes in three launches: Ds is a device array of the scenes' states,
// bmapA / bmapJ map each block of the acceleration / update sweep to
// (scene, particle block within the scene, the block's partial-sum slot in
// the scene's own launch) for lanesA / lanesJ lanes per particle.
// Scenes whose solve has converged return at entry.
void launch_batch_iteration(bool pressure, int lanesA, int lanesJ, const Dev *Ds, const uint4 *bmapA, unsigned nbA,
                            const uint4 *bmapJ, unsigned nbJ, unsigned nscenes, hipStream_t s);
// done[s] = the convergence flag of scene s's current solve.
void launch_batch_done(bool pressure, const Dev *Ds, unsigned nscenes, int *done, hipStream_t s);

class DFSPH {
public:
    explicit DFSPH(const sph_dfsph_params_t &p);
    ~DFSPH();

    sph_dfsph_params_t P;
    double r, hs, V, mass;
    KernelConst K;
    hipStream_t stream = nullptr;
    KernelTimer timer;

    void set_fluid(const float *x, const float *v, size_t n);
    void add_boundary(const float *x, size_t n);
    void set_volume_map_box(const double lo[3], const double hi[3], int invert, double thickness,
                            const unsigned res[3]);
    void add_volume_map(const Shape &shape, const unsigned res[3]);
    void add_volume_map_mesh(const double *vertices, size_t nv, const unsigned *faces, size_t nf, int invert,
                             double thickness, const unsigned res[3]);
    void init();
    void init_if_needed() {
        if (!initialized_) init();
    }
    void reset();
    void emit_particles(const float *x, const float *v, size_t n);
    // Emitter system (EmitterSystem.h/.cpp)
    void add_emitter(const EmitterDesc &e);
    void set_emitter_reuse(bool enable, const double *lo, const double *hi);
    void set_max_emitter_particles(size_t m);
    size_t emitted() const { return emitted_; }
    size_t reused() const { return reused_; }
    const std::vector<EmitterDesc> &emitters() const { return emitters_; }
    // Emitter progress of a resumed state (Emitter::loadState,
    // EmitterSystem::loadState: Emitter.cpp:396-400, EmitterSystem.cpp:128-134).
    void set_emitter_progress(size_t k, double next, unsigned counter);
    void set_emit_counts(size_t emitted, size_t reused) {
        emitted_ = emitted;
        reused_ = reused;
    }
    bool has_states() const { return states_; }
    void step();
    void stage(int s);
    // The step in the parts between its solves (step() = step_begin,
    // divergence solve, step_after_divergence, step_middle, pressure solve,
    // step_after_pressure), for drivers that run the solves of many scenes
    // together. step_begin returns whether the divergence solve runs.
    bool step_begin();
    void step_after_divergence(int iterations);
    void step_middle(bool divergence);
    void step_after_pressure(int iterations);
    int first_chunk(bool pressure) const;  // iterations launched before the first convergence check
    int solve_result(bool pressure, bool read = true);  // the solver counters (read back first)
    // Particles of all scenes stepped together with this one (0: alone).
    void set_company(size_t n) { company_ = n; }
    int lanes_accel() const { return lppA_; }
    int lanes_jacobi() const { return lpp_; }
    Dev device_state() const { return dev(); }
    size_t partial_room() const { return partial_.n; }  // reduction partials (doubles) a launch may write
    bool batchable() const;  // the plain DFSPH step with the reference's warm starts
    bool first_step_pending() const { return !picked_; }  // the next step sets up and picks the lanes per particle
    bool any_xsph() const;   // XSPH acts in some fluid model
    unsigned long long serial() const { return serial_; }  // unique per handle in the process
    // Simulation::setSimulationMethod for this handle: SPH_METHOD_DFSPH,
    // SPH_METHOD_PCISPH (TimeStepPCISPH, pcisph.hip) or SPH_METHOD_IISPH
    // (TimeStepIISPH, iisph.hip)
    void set_method(int m);
    int method() const { return method_; }

    void get_field(const std::string &name, void *host, size_t bytes);
    void set_field(const std::string &name, const void *host, size_t bytes);
    void get_neighbors(int boundary, unsigned *offsets, unsigned *indices, size_t capacity, size_t *nnz);
    void set_warm_start_model(int solver, const float *theta);
    void set_warm_start_policy(int solver, int min_prev_iterations);
    void set_warm_start_mode(int solver, int mode);
    void collect_training(int solver, unsigned stride, size_t capacity);
    void get_training(int solver, float *x, float *t, size_t capacity, size_t *n);
    void counters(sph_dfsph_counters_t *c);
    void set_time(double t, double h);
    void sync();
    size_t n() const { return n_; }

    std::vector<std::unique_ptr<VolumeMap>> vmaps;  // boundary objects, in insertion order

    // RigidBodyObject state of boundary object o (Bender2019 volume maps):
    // position of its reference point, rotation (row-major), velocity and
    // angular velocity; kind 0 at rest (placed by the transform), 1 animated,
    // 2 dynamic (collects the fluid's forces).
    void set_body_motion(unsigned o, const double pos[3], const double R[9], const double vel[3],
                         const double omega[3], int kind);
    // BoundaryModel::getForceAndTorque (+ clearForceAndTorque)
    void body_force(unsigned o, double force[3], double torque[3], bool clear);
    void body_reference(unsigned o, double pos0[3], double *max_dist);

    // Several fluid models (Simulation::numberOfFluidModels): each
    // particle's model (caller order) and five numbers per model: density0,
    // viscosity, viscosityBoundary, xsph, xsphBoundary.
    void set_fluid_models(const unsigned *model, size_t n, const double *materials, unsigned nmodels);
    unsigned fluid_models() const { return models_ ? (unsigned)materials_.size() : 1u; }

private:
    // particle states and emitters
    DBuf<unsigned> pst_, pst2_, mark_, slots_;  // particle states and their permutation target
    DBuf<float4> emit_x_, emit_v_;
    bool states_ = false;  // pst_ holds the particles' states (else all are active)
    std::vector<EmitterDesc> emitters_;
    bool reuse_ = false;
    double reuse_lo_[3] = {-1, -1, -1}, reuse_hi_[3] = {1, 1, 1};
    size_t max_emit_ = 10000, cap_emit_ = 0, emitted_ = 0, reused_ = 0;
    void enable_states();
    void emitter_system_step();
    void emitter_size(const EmitterDesc &e, double *size) const;
    void grow_particles(size_t m);

    size_t n_ = 0;
    unsigned stride_ = 0;
    unsigned long long serial_ = 0;
    bool initialized_ = false, have_lists_ = false;
    unsigned capF_ = 64, capB_ = 64;
    GridDesc grid_{};
    std::vector<float> hx_, hv_, hbx_;  // staged host inputs
    size_t nb_ = 0;
    std::vector<Shape> vm_shapes_;             // staged volume-map objects
    std::vector<std::array<unsigned, 3>> vm_res_;
    unsigned nvm_ = 0;                         // volume maps built

    // device state
    DBuf<float4> x_, v_, v2_, a_, ap_, vdiff_, xc_, vmb_, vmraw_, bx_, dmg_, dmgraw_;
    bool maps() const {  // boundary objects as maps (Bender2019 volume, Koschier2017 density)
        return P.boundary_handling_method == SPH_BOUNDARY_BENDER2019 ||
               P.boundary_handling_method == SPH_BOUNDARY_KOSCHIER2017;
    }
    DBuf<float4> x2_, vdiff2_, xc2_;  // permutation targets
    // moving bodies
    struct BodyMotion {
        int kind = -1;  // -1: never set
        double pos[3], R[9], vel[3], omega[3];
    };
    std::vector<BodyMotion> motion_;  // per boundary object
    // several fluid models
    bool models_ = false;
    DBuf<unsigned> model_, model2_;
    std::vector<std::array<double, 5>> materials_;
    std::vector<unsigned> model_count_;
    bool moving_ = false, dynamic_ = false;
    double body_max_vel_ = 0.0;
    DBuf<float4> vmv_, vmvraw_, body_;
    DBuf<double> bpart_, bforce_;
    std::vector<double> hforce_;  // host copy of the accumulated forces
    void apply_motion();          // motion_ -> map descriptors and the body table
    void body_forces_pressure(bool pressure);
    void body_forces_nonpressure(const Dev &D);
    DBuf<float> rho_, alpha_, radv_, p_, pv_, p2_, pv2_;
    DBuf<unsigned> id_, id2_, nf_, cf_, nb_l_, cb_, bperm_, bstart_;
    DBuf<unsigned> nf16_;    // packed fluid lists (see Dev::nf16)
    bool use16_ = false;     // nf16_ holds the current lists
    DBuf<unsigned> nt16_, tslot_, tcount_;  // tiled fluid lists (see Dev::nt16)
    bool tiled_ = false;     // they hold the current lists
    size_t lists_n_ = 0;     // particles the current lists were built for
    unsigned lists_max_ = 0;  // the longest of them
    bool tiles_known_ = false;  // whether they do has been settled for these lists
    int list_its_ = 0;       // solver iterations on the current lists
    unsigned tiles_over_ = 0, tiles_wait_ = 0;  // overfull tiles when last built, lists since
    bool no_tile_room_ = false;  // their allocation failed at this capacity
    bool tiles_pay() const;
    void build_tiles();
    void ensure_pair_grad();
    DBuf<float4> minv_, cgx_, cgr_, cgp_, cgz_, cgt_;
    DBuf<double> partial_;
    DBuf<Ctl> ctl_;
    DBuf<float> io_;       // field values in id order, on their way from or to the host
    Ctl *hctl_ = nullptr;  // pinned mirror
    CellSorter fsort_, bsort_;
    long long totIt_ = 0, totItV_ = 0, totVisco_ = 0;
    int steps_ = 0, lastIt_ = 2, lastItV_ = 1, lastCg_ = 4;
    int itLast_ = 0, itVLast_ = 0, cgLast_ = 0;
    int capped_ = 0, cappedV_ = 0;
    long long syncs_ = 0;  // host round trips (control-block reads)  // solves stopped at the iteration cap short of the tolerance
    // learned warm start
    bool learned_[2] = {false, false};
    unsigned stride_s_[2] = {0, 0};
    size_t cap_s_[2] = {0, 0};
    DBuf<float> theta_[2], feats_[2], pred_, kprev_, sx_[2], st_[2];
    DBuf<float4> ap2_;
    unsigned soff_ = 0;
    int mode_[2] = {0, 0};  // start of each solve: 0 reference, 1 previous stiffness, 2 network
    bool learn_or_collect(int solver) const { return mode_[solver] != 0 || stride_s_[solver] > 0; }
    bool learned_start(bool pressure);  // true if this solve starts from the network
    bool engaged_[2] = {false, false};   // the current/last solve of each kind started from the network
    int engage_min_[2] = {4, 3};         // engage when the previous solve took at least this many iterations
    int learnedSolves_ = 0, learnedSolvesV_ = 0;
    void collect(bool pressure);
    void ensure_learn_buffers();

    Dev dev() const;
    void alloc_particles();
    void upload_particles(size_t n, const float *x, const float *v, const float4 *xc, const float4 *vdiff,
                          const float *p, const float *pv);
    void upload_ctl_field(size_t off, const void *src, size_t bytes);
    void read_ctl();
    void neighborhood_search();
    void build_lists();
    void volume_maps(const float4 *xin = nullptr, const unsigned *skip = nullptr, const int *stop = nullptr);
    void sweep_init(bool density, bool factor, bool div_setup);
    template <int LPP>
    void sweep_init_l(bool density, bool factor, bool div_setup);
    void div_iteration(bool force);
    void div_finish(bool scale_pv);
    void scale(float *p, int which);
    void clear_accel();
    void viscosity(bool apply_separately);
    // expl: explicit neighbour forces, bit 0 XSPH, bit 1 standard viscosity
    void post_forces(bool clear, bool apply, int expl, bool cfl, bool vupdate, bool scale_pv);
    void pressure_setup();
    void pressure_iteration(bool force);
    void pressure_finish(bool finalize);
    void finalize(bool scale_p, bool update_x);
    // copy_w: copy the stiffness into the position w first (the set-up
    // sweeps of a step write it themselves)
    int run_solver(bool pressure, int already = 0, bool copy_w = true);
    bool mrho_w_ = false;  // position w holds m / rho (within a step's non-pressure forces)
    void mrho_copy();
    // PCISPH
    int method_ = SPH_METHOD_DFSPH;
    double pci_factor_ = 0.0;
    DBuf<float4> predx_, predx2_;  // predicted positions (persistent, sorted with the particles)
    void step_pcisph();
    // IISPH (iisph.hip): d_ii, sum_j d_ij p_j, last pressure, last pressure / rho^2
    DBuf<float4> iid_, iidp_;
    DBuf<float> ilp_, iq_;
    void step_iisph();
    // WCSPH (wcsph.hip): state equation stiffness and exponent
    double wc_k_ = 50.0, wc_gamma_ = 7.0;
    void step_wcsph();

public:
    // TimeStepWCSPH's stiffness and exponent (defaults 50 and 7).
    void set_wcsph(double stiffness, double exponent);

private:
    void stiff_to_w(bool pressure);
    template <bool PRESSURE>
    void iteration_any(bool force);
    void pick_lanes();
    int lpp_ = 1;              // lanes per particle of the Jacobi update and the other sweeps
    int seq_lanes() const { return lpp_ > 4 ? lpp_ : 1; }  // of the sweeps with plain sequential sums at every count
    int lppA_ = 1;             // lanes per particle of the acceleration sweeps (iterations, finish)
    size_t company_ = 0;
    bool picked_ = false, picked_large_ = false, lpp_fixed_ = false;  // picked_large_: at a large count (pick_lanes)

public:
    int lanes_per_particle() const { return lpp_; }
    // 1, 2 or 4 fixes the lanes per particle; 0 leaves them to the rules.
    void set_lanes_per_particle(int lpp);

private:
    int run_cg();
    std::vector<unsigned> ids_host();
};

// Particle files (io.hip): the exporter's particle file, and the fluid part of
// a state file, in the partio BGEO format.
// PCISPH scaling factor of a particle radius r and volume V
// (SimulationDataPCISPH.cpp:40-108).
double pcisph_factor(double r, double V);

void write_particles(DFSPH &s, const std::string &path, const char *fields);
void write_state(DFSPH &s, const std::string &path);
void read_state(DFSPH &s, const std::string &path);

}  // namespace sph
