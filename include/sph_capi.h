/*
 * sph_capi.h -- C-ABI of the MI355X-native DFSPH time step and neighbourhood
 * search (libsph_amd.so, gfx950).
 *
 * Two handle types replace the two C++ interfaces of SPlisHSPlasH v2.16.0 on
 * the hot path:
 *
 *   sph_ns_t     -> SPH::NeighborhoodSearch, the typedef to
 *                   CompactNSearch::NeighborhoodSearch
 *                   (SPlisHSPlasH/NeighborhoodSearch.h:8-14). Member calls
 *                   used by the reference are listed per entry point.
 *   sph_dfsph_t  -> SPH::TimeStepDFSPH (SPlisHSPlasH/DFSPH/TimeStepDFSPH.h:24-76)
 *                   together with the per-particle state it steps
 *                   (FluidModel.h:113-124, SimulationDataDFSPH.h:96-211) and
 *                   the boundary models it reads (BoundaryModel_Akinci2012,
 *                   BoundaryModel_Bender2019).
 *
 * Conventions
 *   - Every entry point returns an int status: SPH_OK (0) or a negative
 *     SPH_ERR_* code; sph_last_error() gives a message for the calling thread.
 *     No C++ exception crosses this boundary.
 *   - Host buffers stay owned by the caller; device memory is owned by the
 *     library. Each handle owns one HIP stream; a handle is not thread-safe.
 *   - Positions are 3 contiguous reals per point (the layout of
 *     std::vector<Vector3r> with Eigen::DontAlign). dtype selects float
 *     (SPH_F32) or double (SPH_F64) input; device arithmetic is FP32 with FP64
 *     reductions.
 *   - There is no CPU fallback: if no gfx950 device is present every
 *     compute entry point returns SPH_ERR_DEVICE.
 */
#ifndef SPH_CAPI_H
#define SPH_CAPI_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define SPH_OK 0
#define SPH_ERR_INVALID  (-1) /* bad argument or handle                     */
#define SPH_ERR_HIP      (-2) /* a HIP runtime call failed                  */
#define SPH_ERR_OOM      (-3) /* device allocation failed                   */
#define SPH_ERR_STATE    (-4) /* call not valid in the handle's state       */
#define SPH_ERR_DEVICE   (-5) /* no usable gfx950 device                    */
#define SPH_ERR_NOTFOUND (-6) /* unknown field name                         */
#define SPH_ERR_RANGE    (-7) /* size beyond a fixed maximum or a capacity  */

#define SPH_F32 0
#define SPH_F64 1

/* Reference enum values (Simulation.h BoundaryHandlingMethods,
 * NonPressureForceRegistration.cpp:52-58). */
#define SPH_BOUNDARY_NONE       (-1)
#define SPH_BOUNDARY_AKINCI2012  0
#define SPH_BOUNDARY_KOSCHIER2017 1  /* density maps of the boundary objects */
#define SPH_BOUNDARY_BENDER2019  2
#define SPH_METHOD_WCSPH         0   /* Simulation simulationMethod values */
#define SPH_METHOD_PCISPH        1
#define SPH_METHOD_IISPH         3
#define SPH_METHOD_DFSPH         4
#define SPH_VISCOSITY_NONE       0
#define SPH_VISCOSITY_STANDARD   1   /* Viscosity_Standard (explicit)        */
#define SPH_VISCOSITY_WEILER2018 6

const char *sph_last_error(void);
/* Library version as MAJOR*10000 + MINOR*100 + PATCH. */
int sph_version(void);
/* Number of visible HIP devices (0 if none); does not fail without a GPU. */
int sph_device_count(int *out);
/* Waits for all work of this process on the current device. */
int sph_device_synchronize(void);

/* ------------------------------------------------------------------------ */
/* Neighbourhood search (the CompactNSearch members the reference calls)    */
/* ------------------------------------------------------------------------ */
typedef struct sph_ns *sph_ns_t;

/* NeighborhoodSearch(Real r, bool erase_empty_cells) -- Simulation.cpp:149 */
int sph_ns_create(double radius, int erase_empty_cells, sph_ns_t *out);
int sph_ns_destroy(sph_ns_t ns);
/* set_radius(Real) -- Simulation.cpp:151 */
int sph_ns_set_radius(sph_ns_t ns, double radius);
int sph_ns_get_radius(sph_ns_t ns, double *out);
/* reset() -- SimulatorBase.cpp:850: forget all point sets. */
int sph_ns_reset(sph_ns_t ns);
/* add_point_set(x, n, is_dynamic, search_neighbors, find_neighbors, user_data)
 * -- FluidModel.cpp:323, BoundaryModel_Akinci2012.cpp:109. The library keeps
 * the caller's pointer (as CompactNSearch does) and reads it on
 * update_point_sets()/find_neighbors(points_changed=1). */
int sph_ns_add_point_set(sph_ns_t ns, const void *x, size_t n, int dtype,
                         int is_dynamic, int search_neighbors,
                         int find_neighbors, void *user_data,
                         unsigned *out_index);
/* resize_point_set(i, x, n) -- FluidModel.cpp:216,737 */
int sph_ns_resize_point_set(sph_ns_t ns, unsigned set, const void *x,
                            size_t n);
/* update_point_sets() -- host-to-device copy of every dynamic set. */
int sph_ns_update_point_sets(sph_ns_t ns);
/* find_neighbors(bool points_changed=true) -- Simulation.cpp:617 */
int sph_ns_find_neighbors(sph_ns_t ns, int points_changed);
/* find_neighbors(Real const* x, vector<vector<unsigned>>&) -- point query
 * (Tools/FoamGenerator/main.cpp:1452). Writes the neighbours of x in `set`
 * into out[0..cap) in ascending order and the total count to *count. */
int sph_ns_query_point(sph_ns_t ns, const double x[3], unsigned set,
                       unsigned *out, unsigned cap, unsigned *count);
/* z_sort() -- Simulation.cpp:626: computes the Morton-order permutation of
 * every dynamic set; sort_field then applies it. */
int sph_ns_z_sort(sph_ns_t ns);
/* PointSet::sort_field<T>(T*) -- permutes a caller array of n elements of
 * elem_bytes bytes in place with the last z_sort() permutation. */
int sph_ns_sort_field(sph_ns_t ns, unsigned set, void *data,
                      size_t elem_bytes);
/* set_active(bool) / set_active(i, search, find) / set_active(i, j, bool)
 * -- Simulation.cpp:713-754 */
int sph_ns_set_active_all(sph_ns_t ns, int active);
int sph_ns_set_active_set(sph_ns_t ns, unsigned set, int search_neighbors,
                          int find_neighbors);
int sph_ns_set_active_pair(sph_ns_t ns, unsigned i, unsigned j, int active);
int sph_ns_is_active_pair(sph_ns_t ns, unsigned i, unsigned j, int *out);
/* n_point_sets(), point_set(i).n_points(), get_user_data() */
int sph_ns_n_point_sets(sph_ns_t ns, unsigned *out);
int sph_ns_n_points(sph_ns_t ns, unsigned set, size_t *out);
int sph_ns_user_data(sph_ns_t ns, unsigned set, void **out);
/* PointSet::n_neighbors(j, i), neighbor(j, i, k), neighbor_list(j, i)
 * -- Simulation.h:456-473. Indices refer to the caller's point order. The
 * list pointer stays valid until the next find_neighbors/z_sort/reset. */
int sph_ns_n_neighbors(sph_ns_t ns, unsigned set_i, unsigned set_j,
                       unsigned i, unsigned *out);
int sph_ns_neighbor(sph_ns_t ns, unsigned set_i, unsigned set_j, unsigned i,
                    unsigned k, unsigned *out);
int sph_ns_neighbor_list(sph_ns_t ns, unsigned set_i, unsigned set_j,
                         unsigned i, const unsigned **out, unsigned *count);
/* Bulk CSR view of all lists of (set_i -> set_j): offsets has n_points+1
 * entries. Same lifetime as sph_ns_neighbor_list. */
int sph_ns_neighbor_csr(sph_ns_t ns, unsigned set_i, unsigned set_j,
                        const unsigned **offsets, const unsigned **indices);

/* Allocation-free search. No counterpart in the reference: it is for callers
 * that cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc). It returns the lists that
 * sph_ns_find_neighbors + sph_ns_neighbor_csr give for one point set that
 * searches itself (same sets, order and indices), computed on device memory:
 *   x          device pointer, 3*n floats (x, y, z per point)
 *   offsets    device pointer, n+1 entries (CSR row offsets, written)
 *   neighbors  device pointer, `capacity` entries (CSR column indices)
 *   *total     host: number of entries (offsets[n]); when it exceeds
 *              `capacity` the call fails with SPH_ERR_RANGE after writing
 *              offsets and *total, so the caller can size the buffer
 *   stream     hipStream_t to run on (NULL: the null stream); the call
 *              returns after the stream has finished its work.
 * Every intermediate lives in one fixed 48 MiB device array per GPU, held
 * from the library's first use on that GPU until the process ends. At most
 * 524,288 points; the cell grid (cells of edge radius over the points'
 * bounding box plus one cell) gets the rest of the array, and a larger
 * grid fails with SPH_ERR_RANGE. All calls on one GPU share the array:
 * the library serialises them per GPU within a process, and a call must
 * not overlap other work that uses its output buffers. */
int sph_ns_find_neighbors_noalloc(const float *x, size_t n, double radius,
                                  unsigned *offsets, unsigned *neighbors,
                                  size_t capacity, size_t *total,
                                  void *stream);

/* ------------------------------------------------------------------------ */
/* DFSPH time step                                                            */
/* ------------------------------------------------------------------------ */
typedef struct sph_dfsph *sph_dfsph_t;

typedef struct sph_dfsph_params {
    double particle_radius;     /* Simulation particleRadius; h = 4r        */
    double density0;            /* FluidModel density0                      */
    double gravity[3];          /* Simulation gravitation                   */
    double time_step_size;      /* TimeManager initial h                    */
    int    cfl_method;          /* 0 off, 1 CFL, 2 CFL + iteration rule     */
    double cfl_factor;
    double cfl_min_time_step_size;
    double cfl_max_time_step_size;
    int    min_iterations;      /* DFSPH.minIterations                      */
    int    max_iterations;      /* DFSPH.maxIterations                      */
    double max_error;           /* DFSPH.maxError, percent                  */
    int    max_iterations_v;    /* DFSPH.maxIterationsV                     */
    double max_error_v;         /* DFSPH.maxErrorV, percent                 */
    int    enable_divergence_solver;
    double xsph;                /* XSPH.xsph                                */
    double xsph_boundary;       /* XSPH.xsphBoundary                        */
    int    viscosity_method;    /* SPH_VISCOSITY_*                          */
    double viscosity;           /* viscosity of the chosen method           */
    double viscosity_boundary;  /* its viscosityBoundary                    */
    int    visco_max_iter;
    double visco_max_error;
    int    boundary_handling_method; /* SPH_BOUNDARY_*                      */
    int    reserved[8];
} sph_dfsph_params_t;

/* Defaults of the reference constructors (Simulation.cpp:66-89,
 * TimeStepDFSPH.cpp:29-41, TimeManager.cpp:12, XSPH.cpp:20,
 * Viscosity_Weiler2018.cpp:21-29). */
void sph_dfsph_default_params(sph_dfsph_params_t *p);

typedef struct sph_dfsph_counters {
    double time;             /* TimeManager time after the last step       */
    double time_step_size;   /* TimeManager h after the last step          */
    double avg_density_err;  /* last pressure iteration, kg/m^3            */
    double avg_divergence_err; /* last divergence iteration                */
    int    iterations;       /* "DFSPH - iterations" (m_iterations)         */
    int    iterations_v;     /* "DFSPH - iterationsV" (m_iterationsV)       */
    int    visco_iterations; /* "Visco iterations" (Eigen CG iters)         */
    int    steps;            /* steps taken since creation                  */
    long long total_iterations;
    long long total_iterations_v;
    long long total_visco_iterations;
    int    max_fluid_neighbors;
    int    max_boundary_neighbors;
    int    flags;            /* bit0: NaN/Inf seen in a reduction           */
    int    learned_particles;   /* particles that kept the learned start in
                                   the last pressure solve                  */
    int    learned_particles_v; /* same, last divergence solve              */
    int    capped_solves;    /* pressure solves that stopped at max_iterations
                                without reaching the tolerance (cumulative)  */
    int    capped_solves_v;  /* same, divergence solves                     */
    int    learned_solves;   /* pressure solves started from the network     */
    int    learned_solves_v; /* divergence solves started from the network   */
    int    lanes_per_particle; /* lanes sharing one particle's neighbour sums
                                  in the Jacobi updates and the other sweeps
                                  (1, 2 or 4; 16 for small counts)          */
    /* Excess of the last iteration: rho0 * mean over particles that keep
     * pressure of the positive residual (s - A p)_i, i.e. expansion the
     * pressure overshoots. The reference's error (above) counts only
     * remaining compression; a solve started from the learned network must
     * bring both below the tolerance. Same units as the errors above. */
    double avg_overpressure_err;
    double avg_overpressure_err_v;
    long long host_syncs;    /* host waits on the device so far (solver
                                chunk ends, list capacity checks)           */
    int    lanes_per_particle_accel; /* same as lanes_per_particle, for the
                                  acceleration sweeps of the solvers        */
    int    packed_lists;     /* 1: the sweeps read the fluid neighbour lists
                                as 16-bit slot differences (every difference
                                of the current lists fits), 0: 32-bit slots */
} sph_dfsph_counters_t;

/* Sub-steps of TimeStepDFSPH::step() (TimeStepDFSPH.cpp:117-249), callable
 * one at a time so a caller can check each against its own reference. */
enum sph_dfsph_stage {
    SPH_STAGE_NEIGHBORHOOD_SEARCH = 0, /* Simulation::performNeighborhoodSearch */
    SPH_STAGE_VOLUME_MAPS        = 1, /* TimeStep::computeVolumeAndBoundaryX  */
    SPH_STAGE_DENSITIES          = 2, /* TimeStep::computeDensities           */
    SPH_STAGE_DFSPH_FACTOR       = 3, /* computeDFSPHFactor                   */
    SPH_STAGE_DIVERGENCE_SETUP   = 4, /* divergenceSolve set-up loop          */
    SPH_STAGE_DIVERGENCE_ITER    = 5, /* one divergenceSolveIteration         */
    SPH_STAGE_DIVERGENCE_FINISH  = 6, /* divergenceSolve finalisation         */
    SPH_STAGE_DIVERGENCE_SOLVE   = 7, /* whole divergenceSolve                */
    SPH_STAGE_CLEAR_ACCEL        = 8, /* TimeStep::clearAccelerations         */
    SPH_STAGE_VISCOSITY          = 9, /* Viscosity_Weiler2018::step           */
    SPH_STAGE_XSPH               = 10,/* XSPH::step                           */
    SPH_STAGE_CFL                = 11,/* Simulation::updateTimeStepSize       */
    SPH_STAGE_UPDATE_VELOCITY    = 12,/* v += h_old a                         */
    SPH_STAGE_PRESSURE_SETUP     = 13,/* pressureSolve set-up loop            */
    SPH_STAGE_PRESSURE_ITER      = 14,/* one pressureSolveIteration           */
    SPH_STAGE_PRESSURE_FINISH    = 15,/* pressureSolve finalisation           */
    SPH_STAGE_PRESSURE_SOLVE     = 16,/* whole pressureSolve                  */
    SPH_STAGE_UPDATE_POSITION    = 17,/* x += h_old v and t += h_old          */
    SPH_STAGE_COUNT              = 18
};

int sph_dfsph_create(const sph_dfsph_params_t *params, sph_dfsph_t *out);
int sph_dfsph_destroy(sph_dfsph_t s);
/* FluidModel::initModel (FluidModel.cpp:285-327): n particles, positions and
 * velocities as 3n floats. Particle i gets id i. */
int sph_dfsph_set_fluid(sph_dfsph_t s, const float *x, const float *v,
                        size_t n);
/* BoundaryModel_Akinci2012::initModel (BoundaryModel_Akinci2012.cpp:77-110)
 * for a static body: n boundary particles, 3n floats. */
int sph_dfsph_add_boundary_particles(sph_dfsph_t s, const float *x, size_t n);
/* With boundary_handling_method SPH_BOUNDARY_KOSCHIER2017 the three calls
 * below add BoundaryModel_Koschier2017 objects instead: field 1 is the
 * density map of SimulatorBase::initDensityMap (SimulatorBase.cpp:
 * 2322-2500: 0.8 times the integral over the support of (1 - 5 d / h) W
 * where the distance d is at most h/5, 26-point Gauss rule per axis), and
 * each step samples rho_b, grad rho_b and the boundary point per particle
 * (TimeStep::computeDensityAndGradient, TimeStep.cpp:349-468).
 *
 * Adds a BoundaryModel_Bender2019 boundary object: the volume map of an
 * axis-aligned box wall (SimulatorBase::initVolumeMap,
 * SimulatorBase.cpp:2566-2704): the signed distance of the box surface
 * (inverted when `invert`, i.e. fluid inside), minus `thickness`, discretised
 * on resolution[0..2] cubic cells over the box grown by 8h + thickness, and
 * the volume field integrated from it. Boundary objects are sampled and
 * summed in the order they were added (TimeStep.cpp:177-222). */
int sph_dfsph_set_volume_map_box(sph_dfsph_t s, const double box_min[3],
                                 const double box_max[3], int invert,
                                 double thickness,
                                 const unsigned resolution[3]);
/* Adds a Bender2019 boundary object for a static sphere: the analytic
 * signed distance |x - centre| - radius (negated when `invert`: fluid
 * inside), minus `thickness`, on resolution[0..2] cells over the sphere's
 * bounding box grown by 8h + thickness. The reference builds the same map
 * from a sphere mesh's distance field (SimulatorBase.cpp:2566-2704). */
int sph_dfsph_add_volume_map_sphere(sph_dfsph_t s, const double centre[3],
                                    double radius, int invert,
                                    double thickness,
                                    const unsigned resolution[3]);
/* Adds a Bender2019 boundary object for a static closed triangle mesh
 * (vertices: 3 doubles each, world coordinates; faces: 3 vertex indices
 * each). The distance field at the grid nodes is the distance to the
 * nearest triangle, negative inside (generalized winding number above 1/2;
 * positive inside when `invert`), minus `thickness`; the volume field
 * integrates the interpolated distance field, as SimulatorBase::
 * initVolumeMap does with Discregrid's (SimulatorBase.cpp:2566-2704). */
int sph_dfsph_add_volume_map_mesh(sph_dfsph_t s, const double *vertices,
                                  size_t n_vertices, const unsigned *faces,
                                  size_t n_faces, int invert, double thickness,
                                  const unsigned resolution[3]);
/* Deferred initialisation (SimulatorBase::deferredInit,
 * StaticBoundarySimulator.cpp:181-199): Akinci boundary volumes
 * (Simulation::updateBoundaryVolume) and device buffers. Called by the first
 * step if not called before. */
int sph_dfsph_init(sph_dfsph_t s);
/* n_steps calls of TimeStepDFSPH::step(). */
int sph_dfsph_step(sph_dfsph_t s, int n_steps);
/* TimeStepDFSPH::reset (TimeStepDFSPH.cpp:710-716, SimulationDataDFSPH.cpp:
 * 64-81): zeroes the solver's per-particle fields (factor, advected density,
 * p / rho^2, p_v / rho^2, pressure acceleration) and the iteration counters.
 * Positions, velocities, densities, time and the viscosity warm start are
 * kept, as in the reference. */
int sph_dfsph_reset(sph_dfsph_t s);
/* Particles activated by an emitter (Emitter.cpp:180-225) followed by
 * TimeStepDFSPH::emittedParticles and resize (TimeStepDFSPH.cpp:723-731,
 * SimulationDataDFSPH.cpp:103-112): appends n particles with positions x and
 * velocities v (3n floats each; v may be null for zero). They get ids
 * num_particles() .. num_particles() + n - 1 and zero stiffness; the other
 * particles keep their state. */
int sph_dfsph_emit_particles(sph_dfsph_t s, const float *x, const float *v,
                             size_t n);
/* Simulation::setSimulationMethod (Simulation.cpp:528-580) for this handle:
 * SPH_METHOD_DFSPH (default); SPH_METHOD_PCISPH, TimeStepPCISPH::step
 * (PCISPH/TimeStepPCISPH.cpp:80-128): the predictor-corrector pressure loop
 * with the scaling factor of SimulationDataPCISPH::init; or SPH_METHOD_IISPH,
 * TimeStepIISPH::step (IISPH/TimeStepIISPH.cpp:91-554): predictAdvection
 * and the relaxed Jacobi solve with omega 0.5. Both use the parameters'
 * min_iterations, max_iterations and max_error (their own defaults: 3 / 2,
 * 100 and 0.01 %). The neighbour search, boundaries, non-pressure forces,
 * CFL, states and emitters are shared. Call before the first step or
 * between steps. */
int sph_dfsph_set_simulation_method(sph_dfsph_t s, int method);
/* SPH_METHOD_WCSPH runs TimeStepWCSPH::step (WCSPH/TimeStepWCSPH.cpp:74-199):
 * the state equation p = stiffness ((rho / rho0)^exponent - 1) on the
 * density clamped to rho0, the pressure accelerations and an explicit
 * integration. TimeStepWCSPH's stiffness and exponent (defaults 50, 7). */
int sph_dfsph_set_wcsph(sph_dfsph_t s, double stiffness, double exponent);

/* Emitter system (SPlisHSPlasH/EmitterSystem.h, Emitter.h). An emitter
 * places a width x height grid of particles (type 0, box) or a disc of width
 * particles across (type 1, circle) at translation + (t - next + h) v along
 * column 0 of the row-major rotation, every 2r / velocity seconds between
 * emit_start_time and emit_end_time, and animates the particles inside its
 * region (Emitter.cpp:89-380). Emission happens at the end of each step,
 * before the time advances (TimeStepDFSPH.cpp:242-248). New particles get
 * the next ids and state 1 (animated) for one step. */
typedef struct sph_emitter {
    int      type;               /* 0 box, 1 circle (Emitter m_type)         */
    unsigned width, height;      /* particles across; height: boxes only     */
    double   translation[3];     /* m_x                                      */
    double   rotation[9];        /* m_rotation, row-major                    */
    double   velocity;           /* m_velocity (> 0)                         */
    double   emit_start_time;    /* m_emitStartTime                          */
    double   emit_end_time;      /* m_emitEndTime (DBL_MAX: none)            */
} sph_emitter_t;
/* EmitterSystem::addEmitter + Emitter::setEmitStartTime/EndTime
 * (EmitterSystem.cpp:93-104, SimulatorBase.cpp:1319-1371). */
int sph_dfsph_add_emitter(sph_dfsph_t s, const sph_emitter_t *e);
/* EmitterSystem::enableReuseParticles / disableReuseParticles
 * (EmitterSystem.cpp:106-117): particles leaving [box_min, box_max] are
 * slowed (x 0.95) and placed again by the next emitter layers. */
int sph_dfsph_set_emitter_reuse(sph_dfsph_t s, int enable,
                                const double box_min[3],
                                const double box_max[3]);
/* nMaxEmitterParticles of Simulation::addFluidModel (Simulation.cpp:686,
 * SimulatorBase.cpp:1267-1273, default 10000): emitters stop adding new
 * particles once this many were added. */
int sph_dfsph_set_max_emitter_particles(sph_dfsph_t s, size_t max_particles);
/* m_numberOfEmittedParticles and m_numReusedParticles (EmitterSystem.h). */
int sph_dfsph_emitter_counts(sph_dfsph_t s, size_t *emitted, size_t *reused);

/* Several fluid models in one step (Simulation::addFluidModel; the DFSPH
 * step loops over the models, TimeStepDFSPH.cpp:117-249). model[i] is the
 * model of particle i (caller order, n = the handle's particle count); five
 * numbers per model: density0, viscosity, viscosityBoundary, xsph,
 * xsphBoundary (its Materials entry; the viscosity method and the particle
 * radius are shared). Densities use each particle's rest density, the
 * pressure acceleration weighs neighbour j by rho0_j / rho0_i (:1321),
 * standard viscosity acts within a model, XSPH across models with the
 * neighbour's mass, and each Jacobi iteration updates the models one after
 * the other, the solve stopping when every model meets its own tolerance
 * (:324-341, :477-495). Up to 8 models; DFSPH with the reference's warm
 * start, without emitters and without Weiler2018 viscosity. */
int sph_dfsph_set_fluid_models(sph_dfsph_t s, const unsigned *model, size_t n,
                               const double *materials, unsigned n_models);

/* Moving boundaries: the RigidBodyObject state of boundary object `obj`
 * (the Bender2019 volume maps in insertion order) that a rigid-body solver
 * sets before each step (RigidBodyObject::setPosition / setRotation /
 * setVelocity / setAngularVelocity, SPlisHSPlasH/RigidBodyObject.h; the
 * reference's BoundarySimulator drives them). position is the current
 * position of the body's reference point (sph_dfsph_get_body_reference),
 * rotation the row-major 3x3 turning the shape's frame into the world's;
 * the map is then looked up at R^T (x - position) + reference point
 * (TimeStep.cpp:245-252). kind: 0 at rest (only placed), 1 animated (moves
 * with velocity + angular_velocity x (x - position), BoundaryModel.h:78-84,
 * in every boundary term and the CFL step, Simulation.cpp:470-479),
 * 2 dynamic (also collects the fluid's forces). DFSPH only; not with
 * Weiler2018 boundary viscosity. */
int sph_dfsph_set_body_motion(sph_dfsph_t s, unsigned obj, const double position[3],
                              const double rotation[9], const double velocity[3],
                              const double angular_velocity[3], int kind);
/* BoundaryModel::getForceAndTorque (+ clearForceAndTorque when clear != 0,
 * BoundaryModel.cpp:36-56): the force and the torque about the body's
 * position that the fluid exerted on a dynamic body since the last clear
 * (pressure forces of both solves, TimeStepDFSPH.cpp:1357-1364; XSPH and
 * standard-viscosity boundary terms, XSPH.cpp:203,
 * Viscosity_Standard.cpp:400-403). FP64 sums. */
int sph_dfsph_get_body_force(sph_dfsph_t s, unsigned obj, double force[3],
                             double torque[3], int clear);
/* The body's reference point where its shape was given (the average of the
 * shape's vertices, SimulatorBase.cpp:2710-2717) and the largest vertex
 * distance from it (the maxDist of SimulatorBase.cpp:2719-2729). */
int sph_dfsph_get_body_reference(sph_dfsph_t s, unsigned obj, double position[3],
                                 double *max_dist);

/* Steps n independent scenes together (no reference counterpart, which
 * steps one scene per SimulatorBase::timeStep, SimulatorBase.cpp:959-1006;
 * the ensemble that generates training data): every handle advances n_steps
 * steps. In batch modes 1 and 2 the two solves of a step run
 * for all scenes at once: each Jacobi iteration is one acceleration sweep
 * and one update over every scene's particles plus one reduction block per
 * scene, scenes grouped by their lanes per particle, converged scenes
 * returning at entry; mode 2 replays the iterations between two convergence
 * checks from captured HIP graphs. The rest of each step runs per scene on
 * its own stream over `threads` host threads (0: up to 16). This needs
 * every scene to run the DFSPH step with the reference's warm starts, not
 * collecting training samples, all with or all without the divergence
 * solver; otherwise, and in mode 0, the handles are shared out over the
 * host threads by particle count and each thread interleaves its scenes
 * step by step. Each scene's results are those of sph_dfsph_step on it
 * alone with the same lanes per particle. When some handle has yet to pick
 * its lanes per particle (its first step after creation or after lanes 0 was
 * set), every handle first takes one step here, one handle at a time, and
 * the mode runs the remaining n_steps - 1. A handle may appear once; the
 * first error of any scene is returned. */
int sph_dfsph_step_batch(sph_dfsph_t *handles, size_t n, int n_steps,
                         int threads);
/* Batch mode of sph_dfsph_step_batch for the process: 0 scene by scene on
 * host threads, 1 batched solves, 2 batched solves replayed from HIP graphs,
 * 3 (default) the faster of 0 and 2 for each set of handles: its first four
 * steps alternate the two, the second step of each is timed, and the faster
 * way runs from then on. No reference counterpart. */
int sph_dfsph_set_batch_mode(int mode);
/* The way mode 3 chose for the last set of handles: 0 or 2, -1 while the
 * first steps are still being timed. No reference counterpart. */
int sph_dfsph_batch_choice(void);
/* One sub-step, see enum sph_dfsph_stage. */
int sph_dfsph_stage(sph_dfsph_t s, int stage);
int sph_dfsph_num_particles(sph_dfsph_t s, size_t *out);
/* Field access by the reference's field names (TimeStepDFSPH.cpp:49-53,
 * FluidModel fields, Viscosity_Weiler2018.cpp:33): "position", "velocity",
 * "acceleration", "density", "factor", "advected density", "p / rho^2",
 * "p_v / rho^2", "pressure acceleration", "velocity difference", "id",
 * "boundary volume", "boundary x", "boundary particle volume",
 * "fluid neighbor count", "boundary neighbor count". Values are float32
 * (uint32 for ids and counts) in particle-id order; bytes must equal
 * n * components * 4. */
int sph_dfsph_get_field(sph_dfsph_t s, const char *name, void *host,
                        size_t bytes);
int sph_dfsph_set_field(sph_dfsph_t s, const char *name, const void *host,
                        size_t bytes);
/* Neighbour lists of the last search, particle-id indexed CSR (fluid->fluid
 * when boundary == 0, fluid->boundary particles when boundary == 1).
 * offsets: n+1 entries; indices: capacity entries; *nnz receives the total. */
int sph_dfsph_get_neighbors(sph_dfsph_t s, int boundary, unsigned *offsets,
                            unsigned *indices, size_t capacity, size_t *nnz);
int sph_dfsph_get_counters(sph_dfsph_t s, sph_dfsph_counters_t *out);
int sph_dfsph_set_time(sph_dfsph_t s, double time, double time_step_size);
/* Per-kernel GPU timing with HIP events on the handle's stream. When
 * enabled, sph_dfsph_kernel_stats reports, for kernel k < *count, its name,
 * launch count and summed milliseconds. */
int sph_dfsph_enable_timing(sph_dfsph_t s, int enable);
/* Restricts timing to the kernels named in the comma-separated list (null
 * or empty: all), so that a timed run records two events per launch of
 * those kernels only. */
int sph_dfsph_time_only(sph_dfsph_t s, const char *names);
/* Lanes per particle of the sweeps: 1, 2 or 4 for all of them, or 0
 * (default) to leave them to a rule on the particle count and the lists, for
 * the acceleration sweeps and for the Jacobi update (which the other sweeps
 * follow). They fix the order of the FP32 neighbour sums. From 65,536
 * particles on the rule is applied at the first sweep and its choice kept
 * until the caller adds particles (sph_dfsph_emit_particles, a longer state
 * file) or sets lanes again; below, one lane's sums are taken, up to 40,960
 * particles (of all scenes stepped together) by 16 lanes that share a
 * particle's pairs. */
int sph_dfsph_set_lanes_per_particle(sph_dfsph_t s, int lanes);
int sph_dfsph_kernel_stats(sph_dfsph_t s, int k, const char **name,
                           long long *launches, double *total_ms,
                           int *count);
int sph_dfsph_reset_kernel_stats(sph_dfsph_t s);
int sph_dfsph_synchronize(sph_dfsph_t s);

/* ------------------------------------------------------------------------ */
/* Learned warm start (no counterpart in the reference): a per-particle MLP   */
/* 6 -> 64 -> 64 -> 1 with SiLU, BF16 MFMA with FP32 accumulation. theta is  */
/* the flat parameter vector W1 (6x64 [in][out]), b1 (64), W2 (64x64), b2     */
/* (64), W3 (64), b3 (1); inputs are rows of 8 floats (6 features + 2 zeros). */
/* ------------------------------------------------------------------------ */
int sph_mlp_num_params(void);
/* y[i] = net(x[i]), host buffers. */
int sph_mlp_forward(const float *theta, const float *x, size_t n, float *y);
/* Mean squared error over the n samples and its gradient (host buffers). */
int sph_mlp_loss_grad(const float *theta, const float *x, const float *t,
                      size_t n, float *grad, float *loss);
/* `steps` Adam steps (lr, beta 0.9/0.999) on minibatches of `batch` rows of
 * a seeded shuffle of the samples; theta is updated in place and the final
 * loss over all samples is returned in *loss. */
int sph_mlp_train(float *theta, const float *x, const float *t, size_t n,
                  int steps, int batch, double lr, unsigned seed, float *loss);

/* Learned warm start inside the time step (no counterpart in the reference;
 * the hook replaces the warm starts of TimeStepDFSPH.cpp:292-296 and
 * :449-453). solver: 0 pressure solve, 1 divergence solve. With a model set
 * (warm-start mode 2), the solve starts from the network's prediction
 * wherever its initial residual is smaller than that of the previous-step
 * start, and then iterates to the same tolerance on the reference's error
 * (remaining compression) and on the overshoot (counters
 * avg_overpressure_err*), which the reference's conservative start keeps
 * near zero by construction. theta == NULL restores the reference's start
 * (mode 0). */
int sph_dfsph_set_warm_start_model(sph_dfsph_t s, int solver,
                                   const float *theta);
/* Start of the solves of `solver` (no reference counterpart): 0 the
 * reference's warm start; 1 the previous step's full stiffness (the
 * reference's start without its factor 1/2 and clamp), kept per particle
 * where it beats the same start masked as the reference masks it; 2 the
 * network's prediction (needs sph_dfsph_set_warm_start_model, which selects
 * it), with the masked previous stiffness as the per-particle fallback. */
int sph_dfsph_set_warm_start_mode(sph_dfsph_t s, int solver, int mode);
/* When to use the better start (no reference counterpart): after a solve from
 * the reference's start, the next solve of the same kind starts from the
 * network if that solve took at least `min_prev_iterations` iterations
 * (defaults: pressure 4, divergence 3); below that the reference's start is
 * already near the solution and the network's extra sweeps cost more than
 * they save. After a solve from the network, the network stays in use
 * unless that solve ended at the minimum iteration count. 0 = always. */
int sph_dfsph_set_warm_start_policy(sph_dfsph_t s, int solver,
                                    int min_prev_iterations);
/* Training-sample collection: after each solve, every `stride`-th particle
 * (rotating offset) contributes its 6 features (rows of 8 floats) and its
 * converged stiffness relative to the step's scale; up to `capacity`
 * samples are kept on the device. stride 0 turns collection off. */
int sph_dfsph_collect_training(sph_dfsph_t s, int solver, unsigned stride,
                               size_t capacity);
/* Copies the collected samples (x: n rows of 8 floats, t: n targets) and
 * clears the buffer; *n receives the number copied. */
int sph_dfsph_get_training(sph_dfsph_t s, int solver, float *x, float *t,
                           size_t capacity, size_t *n);

/* Cubic-spline table kernel (PrecomputedKernel<CubicKernel,10000>,
 * SPHKernels.h:614-691) evaluated on the device for n FP32 offsets r (3n
 * floats): W into w[n], gradW into g[3n]. For kernel checks. */
int sph_kernel_eval(double support_radius, const float *r, size_t n,
                    float *w, float *g);

/* ------------------------------------------------------------------------ */
/* Scene front-end                                                            */
/* ------------------------------------------------------------------------ */
typedef struct sph_scene *sph_scene_t;

/* SceneLoader::readScene (SPlisHSPlasH/Utilities/SceneLoader.cpp:13-150)
 * for what this time step runs. Read: "Configuration" (particleRadius,
 * timeStepSize, gravitation, cflMethod, cflFactor, cflMin/MaxTimeStepSize,
 * boundaryHandlingMethod, simulationMethod 4 (DFSPH) with the "DFSPH"
 * section, 1 (PCISPH) or 3 (IISPH) with their sections, or 0 (WCSPH) with
 * its "WCSPH" section), the fluid's "Materials"
 * entry (density0, viscosityMethod 0/1/6 with its "Standard viscosity" or
 * "Weiler et al. 2018" section, the "XSPH" section), "FluidBlocks" sampled
 * as SimulatorBase::createFluidBlocks (Simulator/SimulatorBase.cpp:
 * 1418-1516) with their initial velocities (:1079-1093), "FluidModels"
 * from .bgeo particle files after them (R (s x) + t, then the initial
 * velocities; :1095-1260), and static
 * "RigidBodies" from OBJ meshes (Bender2019 / Koschier2017: one volume or
 * density map each with mapInvert / mapThickness / mapResolution, analytic
 * for an axis-aligned box or a sphere, a mesh map otherwise; Akinci2012:
 * surfaces sampled at 2r, any closed mesh included), and "Emitters" (SimulatorBase::createEmitters,
 * SimulatorBase.cpp:1286-1384: width, height, translation, rotationAxis,
 * rotationAngle, velocity, type, emitStartTime, emitEndTime; the fluid
 * material's maxEmitterParticles, emitterReuseParticles, emitterBoxMin/Max;
 * with Bender2019 or Koschier2017 each emitter also gets its housing as a
 * static mesh body after the scene's bodies). Other keys that do not change the simulation
 * are ignored; anything that would (dynamic bodies, fluid models from
 * files, other methods, several fluid ids) fails with SPH_ERR_INVALID
 * naming the key. Relative geometry paths are resolved against the scene
 * file's folder. */
int sph_scene_load(const char *path, sph_scene_t *out);
int sph_scene_destroy(sph_scene_t s);
int sph_scene_params(sph_scene_t s, sph_dfsph_params_t *params);
int sph_scene_counts(sph_scene_t s, size_t *n_fluid,
                     size_t *n_boundary_particles, int *n_bodies);
/* Fluid positions and velocities (3 floats each, block by block in the
 * reference's sampling order) and Akinci boundary particles; any pointer
 * may be null. */
int sph_scene_particles(sph_scene_t s, float *x, float *v, float *boundary_x);
/* Body k: kind 0 box (lo, hi), 1 sphere (centre, radius) or 2 mesh (lo, hi:
 * its bounding box), and its map settings. */
int sph_scene_body(sph_scene_t s, int k, int *kind, double lo[3], double hi[3],
                   double centre[3], double *radius, int *invert,
                   double *thickness, unsigned resolution[3]);
/* The world-space triangles of a mesh body (kind 2): counts first (null
 * arrays), then 3 doubles per vertex and 3 indices per face. */
int sph_scene_body_mesh(sph_scene_t s, int k, double *vertices,
                        size_t *n_vertices, unsigned *faces, size_t *n_faces);
/* Emitter k of the scene, and the fluid's emitter settings. */
int sph_scene_emitter(sph_scene_t s, int k, sph_emitter_t *out);
int sph_scene_emitter_settings(sph_scene_t s, int *n_emitters,
                               size_t *max_emitter_particles, int *reuse,
                               double box_min[3], double box_max[3]);
/* The scene's simulationMethod and its "WCSPH" section's stiffness and
 * exponent (defaults 50 and 7). */
int sph_scene_simulation_method(sph_scene_t s, int *method,
                                double *wcsph_stiffness, double *wcsph_exponent);
/* A DFSPH handle with the scene's parameters, fluid, boundaries and
 * emitters. */
int sph_scene_create_dfsph(sph_scene_t s, sph_dfsph_t *out);

/* ------------------------------------------------------------------------ */
/* Particle files (partio BGEO)                                              */
/* ------------------------------------------------------------------------ */
/* ParticleExporter_Partio::writeParticlesPartio
 * (Simulator/Exporter/ParticleExporter_Partio.cpp): the particles in
 * particle-id order as a gzip-compressed BGEO file with the position, "id"
 * and the ';'-separated fields (the scene's "particleAttributes", e.g.
 * "velocity;density"; names as in sph_dfsph_get_field). */
int sph_dfsph_write_particles(sph_dfsph_t s, const char *path,
                              const char *fields);
/* SimulatorBase::saveState / loadState (SimulatorBase.cpp:1689-1872) for the
 * fluid: <prefix>_particle_Fluid.bgeo holds the fields the reference stores
 * (writeFluidParticlesState, :2062-2128: id, state, object_id, position,
 * velocity, p / rho^2, p_v / rho^2 and, with Weiler2018, velocity
 * difference), readable by the reference; <prefix>.json holds the time and
 * time step size (the reference keeps those in its own .bin). Loading sets
 * every field of the particle file that the handle has (point i to particle
 * i, readFluidParticlesState :2130-2190) and the time; the particle count
 * must match. */
int sph_dfsph_save_state(sph_dfsph_t s, const char *prefix);
int sph_dfsph_load_state(sph_dfsph_t s, const char *prefix);

/* The file format itself: BGEO version 5 as partio writes it (big-endian,
 * gzip; point position plus point attributes of type 0 float, 1 int or
 * 5 vector). Reading accepts plain or gzip files. */
typedef struct sph_bgeo *sph_bgeo_t;
int sph_bgeo_open(const char *path, sph_bgeo_t *out);
int sph_bgeo_close(sph_bgeo_t f);
int sph_bgeo_count(sph_bgeo_t f, size_t *n_points, int *n_attributes);
int sph_bgeo_attribute(sph_bgeo_t f, int k, const char **name, int *type,
                       int *size);
/* Attribute data (n_points * size 32-bit values), or "position" (3 floats
 * per point). */
int sph_bgeo_data(sph_bgeo_t f, const char *name, void *out, size_t bytes);
int sph_bgeo_write(const char *path, size_t n_points, const float *position,
                   int n_attributes, const char *const *names,
                   const int *types, const int *sizes,
                   const void *const *data);

#ifdef __cplusplus
}
#endif
#endif /* SPH_CAPI_H */
