/*
 * pbd.h - C-ABI of the MI355X-native position-based-fluids (PBF) step.
 *
 * This is the drop-in boundary for the per-frame simulation step of
 * niklasandersson/PBD-Simulation-Framework-CUDA.  In the reference the step is
 * reached through
 *   - Cuda_Computable::compute()           PBD-Simulation-Framework-CUDA/src/cuda/Cuda_Computable.h:8-18
 *   - Fluid::Fluid / ~Fluid / compute()     PBD-Simulation-Framework-CUDA/src/app/simulation/Fluid.cu:4-97
 *   - Simulation::step()                    PBD-Simulation-Framework-CUDA/src/app/Simulation.cu:16-19
 *   - the argument-less cudaCall*() stage functions declared in
 *     PBD-Simulation-Framework-CUDA/src/app/simulation/kernel/Kernels.h:18-43
 * with parameters pulled from the Config singleton (src/parser/Config.h:21-32)
 * and particle buffers owned by OpenGL (src/app/rendering/Particles.cc:4-147).
 * Here the library owns device memory, parameters travel in a POD struct,
 * and every call returns a status code (0 = OK); no exception crosses the ABI.
 *
 * Particle-buffer layout (kept from the reference, kernel/Globals.h:5-13,129-132):
 * four float4 arrays positions4 / predictedPositions4 / velocities4 / colors4,
 * particle i at element i (the reference's texel (i mod W, i div W) of a
 * W x W RGBA32F texture is the same linear float4 array).  After each step the
 * particles are stored in the step's sorted (cell-id, previous-index) order, as
 * in the reference, which reorders its surfaces every frame (SortReorder.h:86-129).
 *
 * Threading: one context is bound to one HIP stream and is not re-entrant;
 * callers serialize, like the reference's single simulation thread.
 */
#ifndef PBD_PBD_H
#define PBD_PBD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PBD_ABI_VERSION 1

/* ---- status codes ------------------------------------------------------ */
enum {
  PBD_OK = 0,
  PBD_ERR_INVALID = 1,     /* bad argument or parameter out of range          */
  PBD_ERR_CAPACITY = 2,    /* particle capacity exceeded (reference ignores it, Communication.h:631,642) */
  PBD_ERR_HIP = 3,         /* a HIP runtime call failed                         */
  PBD_ERR_CONFIG = 4,      /* config.txt missing, malformed or key not found    */
  PBD_ERR_NONFINITE = 5,   /* NaN/Inf found by pbd_check_finite                 */
  PBD_ERR_UNSUPPORTED = 6, /* feature not available in this build             */
  PBD_ERR_NOMEM = 7,       /* host or device allocation failed                  */
  PBD_ERR_IO = 8           /* a file could not be written                       */
};

/* ---- kernel variants (Density.kernelVariant) ---------------------------- */
enum {
  PBD_KERNEL_REFERENCE = 0, /* literal reference formulas, kernel/Density.h:14-42 */
  PBD_KERNEL_TEXTBOOK = 1   /* Macklin & Mueller 2013 PBF with Mueller 2003 kernels */
};

/*
 * pbd_params - POD mirror of the reference's config.txt key set.
 * Replaces SimulationParameters + initializeFrame()'s Config reads
 * (kernel/Globals.h:39-79, kernel/Initialize.h:20-71).  Each field names the
 * config key it mirrors; keys marked "new" are additions with defaults that
 * reproduce the reference.
 */
typedef struct pbd_params {
  /* Application.Cuda */
  uint32_t threads_per_block;          /* Application.Cuda.threadsPerBlock (launch block size) */
  /* Application.OpenGL.Textures */
  uint32_t texture_width;              /* Application.OpenGL.Textures.width; capacity = width^2 */
  /* Application.Simulation.Active.* (stage gates, Fluid.cu:21-95) */
  int32_t active_apply_forces;
  int32_t active_find_contacts;
  int32_t active_find_neighbours;
  int32_t active_compute_lambda;
  int32_t active_compute_delta_positions;
  int32_t active_apply_delta_positions;
  int32_t active_update_positions;
  int32_t active_compute_omegas;
  int32_t active_compute_vorticity;
  int32_t active_compute_viscosity;
  /* Application.Simulation.Collision */
  int32_t collision_type;              /* 0 = per-contact push, 1 = batched pair solver */
  uint32_t kernel_width_neighbours;    /* neighbour stencil half-width in cells */
  uint32_t max_collision_batches;
  float stiffness;
  /* Application.Simulation.Density */
  float k_scorr;
  float kernel_width_spiky;            /* multiple of the particle diameter */
  int32_t n_scorr;
  float q_scorr;                       /* multiple of the spiky kernel width */
  float rest_density;
  float relaxation;                    /* new: epsilon in lambda (reference hard-codes 1e-4) */
  int32_t rest_density_from_lattice;   /* new: rest density from the spawn lattice */
  int32_t kernel_variant;              /* new: PBD_KERNEL_REFERENCE / PBD_KERNEL_TEXTBOOK */
  /* Application.Simulation.Enclosure */
  float enclosure_position_damping;
  float enclosure_velocity_damping;
  float bounds_min[3];                 /* Enclosure.X|Y|Z.min */
  float bounds_max[3];                 /* Enclosure.X|Y|Z.max */
  /* Application.Simulation.Forces */
  float delta_t;                       /* frame time step */
  float gravity;
  uint32_t substeps;                   /* new: substeps per frame (dt = delta_t / substeps) */
  /* Application.Simulation.Iterations */
  uint32_t solver_iterations;
  uint32_t stabilization_iterations;
  /* Application.Simulation.Particles */
  uint32_t max_neighbours_per_particle;
  float particle_radius;
  uint32_t box_width;                  /* Particles.Box.width  (lattice count along x) */
  uint32_t box_height;                 /* Particles.Box.height (along y) */
  uint32_t box_depth;                  /* Particles.Box.depth  (along z) */
  float box_spacing;
  int32_t box_spawn_in_the_beginning;
  float box_origin[3];                 /* new: reference spawns at (30, 32, 30), Particles.cc:197,205 */
  float box_jitter;                    /* new: uniform jitter half-width per axis */
  uint32_t box_seed_lo;                /* new: 64-bit seed of the jitter RNG, low word */
  uint32_t box_seed_hi;                /* new: high word */
  /* Application.Simulation.Viscosity */
  float c_viscosity;
  float kernel_width_poly;             /* absolute */
  /* Application.Simulation.Vorticity */
  float e_vorticity;
  /* Application.Simulation.Grid (new) */
  float grid_cell_size;                /* <= 0 selects the particle diameter (reference: 1.0 = 2r) */
  float grid_origin[3];
  uint32_t grid_dims[3];               /* cells per axis, each in [1, 1024]; reference 128^3 */
  /* Application.Cuda.tileBits (new): neighbour passes on LDS tiles of 2^tileBits
   * Morton-aligned cells (5 = 2x4x4, 6 = 4x4x4) or per particle (0) */
  uint32_t tile_bits;
  /* Unified phase (new, beyond the reference: it has no friction and no solid
   * phase).  Particles of phase PBD_PHASE_SOLID are granular: no density
   * constraint, vorticity or XSPH; contacts with them carry position-based
   * friction (static mu_s, kinetic mu_k; Macklin et al. 2014, eq. 24-25). */
  float friction_static;               /* Collision.frictionStatic  (mu_s, 0 = no friction) */
  float friction_kinetic;              /* Collision.frictionKinetic (mu_k) */
  float box_solid_fraction;            /* Particles.Box.solidFraction: share of the box spawned solid */
  float box_solid_radius;              /* Particles.Box.solidRadius: radius of the seeded solid spheres */
  /* Application.Cuda.autotune (new): 1 = choose the launch shape by timing
   * trial steps (pbd_autotune) before the first step of a context and at the
   * creation of a batch; choices are cached per workload key */
  uint32_t autotune;
} pbd_params;

/* Device pointers of one context (valid until the next pbd_step / add / clear). */
typedef struct pbd_buffers {
  void* positions4;           /* float4[capacity] */
  void* predicted_positions4; /* float4[capacity] */
  void* velocities4;          /* float4[capacity] */
  void* colors4;              /* float4[capacity] */
  void* external_forces4;     /* float4[capacity]: vorticity force carried to the next step */
  uint32_t num_particles;
  uint32_t capacity;
} pbd_buffers;

/* Buffer selectors for pbd_download / pbd_upload. */
enum {
  PBD_BUF_POSITIONS = 0,        /* float4, positions4 */
  PBD_BUF_PREDICTED = 1,        /* float4, predictedPositions4 */
  PBD_BUF_VELOCITIES = 2,       /* float4, velocities4 */
  PBD_BUF_COLORS = 3,           /* float4, colors4 */
  PBD_BUF_EXTERNAL_FORCES = 4,  /* float4, d_externalForces */
  PBD_BUF_DENSITIES = 5,        /* float,  density of the first solver iteration */
  PBD_BUF_LAMBDAS = 6,          /* float,  d_lambdas (last solver iteration) */
  PBD_BUF_CELL_IDS = 7,         /* uint32, sorted cell ids (d_cellIds_out) */
  PBD_BUF_PARTICLE_IDS = 8,     /* uint32, sorted previous indices (d_particleIds_out) */
  PBD_BUF_CELL_STARTS = 9,      /* uint32[table], d_cellStarts, empty = 0xFFFFFFFF */
  PBD_BUF_CELL_ENDINGS = 10,    /* uint32[table], d_cellEndings, empty = N */
  PBD_BUF_NEIGHBOUR_COUNTERS = 11, /* uint32, d_neighbourCounters */
  PBD_BUF_CONTACT_COUNTERS = 12,   /* uint32, d_contactCounters */
  PBD_BUF_OMEGAS = 13,          /* float4 (w unused), d_omegas */
  PBD_BUF_DELTA_POSITIONS = 14, /* float4, d_deltaPositions of the last iteration */
  PBD_BUF_PHASES = 15,          /* uint32, PBD_PHASE_* per particle (new; uploadable) */
  PBD_BUF_COUNT = 16
};

/* ---- parameters / config.txt (host only; no GPU needed) ---------------- */

/* sizeof(pbd_params), for bindings that mirror the struct. */
size_t pbd_params_size(void);
/* Fill with the values of the reference's shipped config.txt. */
int pbd_params_default(pbd_params* out);
/* Parse a config.txt (reference grammar: scopes, key = value;, arrays,
 * strings, // and block comments, #include, #define/#undef, true/false)
 * and fill *out; keys absent from the file keep their pbd_params_default value.
 * Replaces Config::getInstance()/getValue (src/parser/Config.h:21-32,107-111). */
int pbd_params_load(const char* path, pbd_params* out, char* err, size_t err_len);
/* Like pbd_params_load but starts from *inout and only overwrites the keys
 * present in the file (no missing-key error). */
int pbd_params_merge(const char* path, pbd_params* inout, char* err, size_t err_len);
/* Set one key by dotted path with the reference console's range checks
 * (kernel/Communication.h:440-624). */
int pbd_params_set(pbd_params* p, const char* key, const char* value, char* err, size_t err_len);
/* Read one key by dotted path as text. */
int pbd_params_get(const pbd_params* p, const char* key, char* buf, size_t buf_len);
/* Write the parameters as config.txt text (console command 'w',
 * src/parser/ConfigParser.h:241-247, ConfigObject.h:70-95).  Returns the needed size in *needed. */
int pbd_params_write(const pbd_params* p, char* buf, size_t buf_len, size_t* needed);
/* Generate the spawn lattice of Particles.Box (src/app/rendering/Particles.cc:189-222):
 * point (i,j,k) at box_origin + spacing*(i,j,k) + jitter, i over width (x),
 * j over height (y), k over depth (z), index (i*height + j)*depth + k;
 * v = 0; colour from the seeded RNG with w = 1.  Any output pointer may be NULL. */
/* Phases of the particles pbd_generate_box spawns, in the same order: the
 * lattice points inside seeded spheres of radius Box.solidRadius are
 * PBD_PHASE_SOLID until Box.solidFraction of them are (spheres may overlap). */
enum { PBD_PHASE_FLUID = 0, PBD_PHASE_SOLID = 1 };
int pbd_generate_phases(const pbd_params* p, uint32_t* phases, uint32_t capacity, uint32_t* n_out);
int pbd_generate_box(const pbd_params* p, float* pos4, float* vel4, float* col4,
                     uint32_t capacity, uint32_t* n_out);
/* Rest density of the spawn lattice under the selected kernel variant. */
int pbd_lattice_rest_density(const pbd_params* p, double* out);
/* Morton code of integer cell coordinates (kernel/Hash.h:10-29; x at bit 3b+2,
 * y at 3b+1, z at 3b), and the cell id / cell coordinates of a position with
 * the FP32 arithmetic the step uses (same code as the GPU path). */
uint32_t pbd_morton_encode(uint32_t x, uint32_t y, uint32_t z);
int pbd_cell_key(const pbd_params* p, const float pos[3], uint32_t* key, uint32_t ijk[3]);

/* ---- context ------------------------------------------------------------ */

typedef struct pbd_ctx pbd_ctx;

/* Create a context on the current HIP device.  max_particles = 0 selects
 * texture_width^2 (Particles.cc:11-12).  Replaces cudaInitializeKernels
 * (kernel/Initialize.h:122-130) plus the GL buffer allocation of Particles. */
int pbd_create(const pbd_params* p, uint32_t max_particles, pbd_ctx** out);
/* Replace the parameters; applied at the next step (initializeFrame,
 * kernel/Initialize.h:20-86). */
int pbd_set_params(pbd_ctx* ctx, const pbd_params* p);
int pbd_get_params(pbd_ctx* ctx, pbd_params* out);
/* Append n particles (addParticlesCallback, kernel/Communication.h:637-655).
 * Returns PBD_ERR_CAPACITY instead of silently ignoring an overflow.
 * vel4 / col4 may be NULL (zero velocity, white). */
int pbd_add_particles(pbd_ctx* ctx, uint32_t n, const float* pos4, const float* vel4,
                      const float* col4);
/* One particle at pos with velocity 50*dir, red (addParticleCallback,
 * kernel/Communication.h:22-38,626-635). */
int pbd_add_particle(pbd_ctx* ctx, const float pos[3], const float dir[3]);
/* Spawn the Particles.Box lattice (console 's', Particles.cc:167-170). */
int pbd_spawn_box(pbd_ctx* ctx);
/* N = 0 (clearParticlesCallback, kernel/Communication.h:657-660). */
int pbd_clear_particles(pbd_ctx* ctx);
/* Advance `frames` frames; each frame is `substeps` calls of the step with
 * dt = delta_t / substeps (Fluid::compute, Fluid.cu:14-97).  Stream-ordered:
 * returns after enqueueing; call pbd_sync to wait (Simulation.cu:18). */
int pbd_step(pbd_ctx* ctx, uint32_t frames);
/* Exactly one call of the step (one substep, dt = delta_t / substeps):
 * Fluid::compute (Fluid.cu:14-97). */
int pbd_compute(pbd_ctx* ctx);
/* Same as pbd_step but replays a captured hipGraph of one substep. */
int pbd_step_graph(pbd_ctx* ctx, uint32_t frames);
int pbd_sync(pbd_ctx* ctx);
int pbd_num_particles(pbd_ctx* ctx, uint32_t* n_out);
int pbd_get_buffers(pbd_ctx* ctx, pbd_buffers* out);
/* Synchronous host copies of one buffer (PBD_BUF_*); bytes must not exceed
 * the buffer size.  Upload of PBD_BUF_POSITIONS..PBD_BUF_EXTERNAL_FORCES and
 * PBD_BUF_PHASES only. */
int pbd_download(pbd_ctx* ctx, int which, void* dst, size_t bytes);
int pbd_upload(pbd_ctx* ctx, int which, const void* src, size_t bytes);
/* Size in bytes of buffer `which` for the current particle count. */
int pbd_buffer_bytes(pbd_ctx* ctx, int which, size_t* bytes);
/* Scan positions/velocities for NaN/Inf; PBD_ERR_NONFINITE if any. */
int pbd_check_finite(pbd_ctx* ctx, uint32_t* bad_count);
/* Per-stage timing with HIP events on the context stream (0 = off). */
int pbd_set_timing(pbd_ctx* ctx, int enabled);
/* Stage names and accumulated milliseconds / launch counts since the last
 * reset; returns the number of stages in *count. */
int pbd_get_timings(pbd_ctx* ctx, const char** names, double* ms, uint64_t* launches,
                    uint32_t cap, uint32_t* count);
int pbd_reset_timings(pbd_ctx* ctx);
/* Cumulative work counters since creation or the last reset (diagnostics of
 * the neighbour passes; no counterpart in the reference):
 *   PBD_COUNTER_LIST_BUILDS    lambda and omega passes (each builds or keeps
 *                              the neighbour lists of its tiles)
 *   PBD_COUNTER_LIST_CARRIES   particle-passes that kept the lists their tile
 *                              built in an earlier pass of the substep (tiles
 *                              that carry their lists, halo within the skin)
 *   PBD_COUNTER_LIST_RESCANS   particle-passes of carrying tiles whose halo
 *                              moved too far: their lists were rebuilt
 *   PBD_COUNTER_UNLISTED_LONG  particle-builds with more pairs in range than a
 *                              list holds
 *   PBD_COUNTER_UNLISTED_CAP   particle-builds whose 27-cell count exceeds
 *                              maxNeighboursPerParticle (the truncated order of
 *                              the reference applies: scanned per particle)
 *   PBD_COUNTER_UNLISTED_BLOCK particle-builds in cell blocks whose halo does
 *                              not fit in LDS (scanned per particle)
 * An unlisted particle is scanned again by the pass that would read its list.
 * The reverse passes (pbd_adj_backward, from 2^15 particles on) count their
 * per-particle neighbour lists of each position set:
 *   PBD_COUNTER_ADJ_LISTED_TILE   lists built on the LDS tiles
 *   PBD_COUNTER_ADJ_LISTED_GLOBAL lists built per particle from the cell table
 *                                 (blocks whose halo exceeds the tile capacity)
 *   PBD_COUNTER_ADJ_SCANNED       particles with more candidates in range than
 *                                 a list holds (their passes scan the stencil)
 *   PBD_COUNTER_ADJ_FROM_FORWARD  of the tile lists, those taken from the lists
 *                                 the recomputed forward's passes built for the
 *                                 same positions (no distance tests)
 * Writes min(cap, PBD_COUNTER_COUNT) values; *count = PBD_COUNTER_COUNT. */
enum {
  PBD_COUNTER_LIST_BUILDS = 0,
  PBD_COUNTER_UNLISTED_LONG = 1,
  PBD_COUNTER_UNLISTED_CAP = 2,
  PBD_COUNTER_UNLISTED_BLOCK = 3,
  PBD_COUNTER_ADJ_LISTED_TILE = 4,
  PBD_COUNTER_ADJ_LISTED_GLOBAL = 5,
  PBD_COUNTER_ADJ_SCANNED = 6,
  PBD_COUNTER_LIST_CARRIES = 7,
  PBD_COUNTER_LIST_RESCANS = 8,
  PBD_COUNTER_ADJ_FROM_FORWARD = 9,
  PBD_COUNTER_COUNT = 10
};
int pbd_get_counters(pbd_ctx* ctx, uint64_t* values, uint32_t cap, uint32_t* count);
int pbd_reset_counters(pbd_ctx* ctx);
/* ---- Headless frame output ----
 * Replaces the GL renderer as the step's output consumer (src/app/Engine.cu:66-72
 * renders after each Simulation::step).  The renderer draws particle i from
 * texel (i % width, i / width) of the positions4 / colors4 textures
 * (src/app/rendering/Particles.cc:266-274, shader/particles/
 * particleSpriteGeom.vert:35-41); the files keep that index order.
 *   PBD_OUT_RAW         32-byte header {"PBDF", 1, n, texture width, frame, 0, 0, 0}
 *                       (u32 LE), then n float4 positions4, then n float4 colors4
 *   PBD_OUT_PLY_ASCII   PLY, vertex i = particle i: x y z and the renderer's
 *   PBD_OUT_PLY_BINARY  shade mix((0.95,0.97,0.97), (0,0,1), colors4.x^(1/6)) as uchar rgb */
enum { PBD_OUT_RAW = 0, PBD_OUT_PLY_ASCII = 1, PBD_OUT_PLY_BINARY = 2 };
/* The context's current positions4 / colors4 (texture width = Textures.width). */
int pbd_write_frame(pbd_ctx* ctx, const char* path, int format, uint32_t frame);
/* The same from host arrays (colors4 NULL = white); errors: pbd_last_error(NULL). */
int pbd_write_frame_arrays(const char* path, int format, uint32_t frame, uint32_t n, uint32_t texture_width,
                           const float* positions4, const float* colors4);

/* ---- Reverse mode (no counterpart in the reference) ----
 * Gradients of a loss L(x_T, v_T) of the state after `frames` frames
 * (frames x substeps computes of Fluid::compute, src/app/simulation/Fluid.cu:14-97)
 * with respect to the initial velocities, the rest density and the relaxation
 * eps (Density.relaxation).  Supported: kernelVariant textbook, collisionType 0
 * with at most one stabilization iteration, every Active.* stage on, plain
 * (not batched) contexts; otherwise PBD_ERR_UNSUPPORTED.  Solid particles and
 * friction (PBD_BUF_PHASES, Collision.friction*) are differentiated too: the
 * phase masks, and the friction through p* and x of each iteration (the
 * derivative of the sticking or sliding branch the forward took).
 *
 * pbd_adj_forward runs the frames (one graph launch per substep) and keeps a
 * checkpoint of the state (positions, velocities, external forces, and the
 * phases of a phased context; 48 B per particle, +4) at the start of every
 * k_ckpt-th frame.  The context is left in the final state, in its final
 * particle order. */
int pbd_adj_forward(pbd_ctx* ctx, uint32_t frames, uint32_t k_ckpt);
/* For each particle of the final order (count <= number of particles), its
 * index in the order of the state pbd_adj_forward started from. */
int pbd_adj_ids(pbd_ctx* ctx, uint32_t* initial_index, size_t count);
/* dL_dx, dL_dv: float4 per particle (w ignored) in the final order, NULL = 0.
 * Outputs (NULL = not wanted): dL_dv0 and dL_dx0, float4 per particle in the
 * initial order (w = 0); dL_drho0 and dL_deps, scalars.  Each segment of
 * k_ckpt frames is recomputed from its checkpoint while its steps are recorded
 * (about 104 + 20 x solverIterations bytes per particle and step; phases add 4,
 * friction 16 x solverIterations), then the
 * reverse kernels run over the same sorted neighbour structure (from 2^15
 * particles on with neighbour lists per position set: 288 B per particle,
 * allocated by pbd_adj_forward, taken from the tile lists the recomputation
 * built, which the records keep when the memory is there: 64 + 128 x
 * (solverIterations + 1) B per particle and step; otherwise rebuilt).  The host
 * arrays are copied through pinned memory that pbd_adj_forward allocates (64 B
 * per particle; without it, directly).  The context
 * is left as pbd_adj_forward left it.  PBD_ERR_UNSUPPORTED if a neighbour list
 * reached maxNeighboursPerParticle (a capped neighbour relation is not
 * symmetric). */
int pbd_adj_backward(pbd_ctx* ctx, const float* dL_dx, const float* dL_dv, float* dL_dv0, float* dL_drho0,
                     float* dL_deps, float* dL_dx0);
/* Where the reverse passes' neighbour lists come from (from 2^15 particles on):
 * from_forward = 1 (the default), from the tile lists the recorded steps built
 * (their records keep them: 64 + 128 x (solverIterations + 1) B per particle
 * and step, when the forward runs 2^5-cell tiles); 0, built by the reverse
 * passes themselves (no such memory).  The lists, and so the gradients, are
 * the same either way.  Takes effect at the next pbd_adj_forward. */
int pbd_adj_set_lists(pbd_ctx* ctx, int from_forward);

/* ---- Launch shapes and the autotuner (no counterpart in the reference, whose
 * launch shape is Application.Cuda.threadsPerBlock alone: kernel/Initialize.h:73-85,
 * kernel/Globals.h:117-120).  A shape changes how the step is launched, never
 * what it computes: the sort, the tiles and the per-particle kernels produce
 * the same results under every shape. */
typedef struct pbd_launch_shape {
  uint32_t threads_per_block; /* per-particle kernels: 64 .. 1024, a multiple of 64 */
  uint32_t tile_bits;         /* neighbour-pass tiles of 2^tile_bits cells: 5 or 6 (0 = per particle) */
  uint32_t sort_items;        /* onesweep tile of 256 x sort_items keys: 4, 8, 16 (0 = by particle count) */
  uint32_t small_tile_max;    /* blocks of at most this many particles take one wave each: 0 .. 64
                                 (32 and more: of up to 64); a block whose halo does not fit a
                                 wave's tile takes a workgroup all the same (up to 2^16 particles:
                                 one of more than 8).  Until a shape is set, by particle count: 0 up to 2^16, 32 below 2^21, else 64 */
  uint32_t stride_grid;       /* workgroups of the capped tile grid (batches): a multiple of 32 */
  uint32_t list_skin_pct;     /* tile neighbour lists: skin in percent of the list radius, 0 .. 50
                                 (0: every lambda and omega pass rebuilds its lists) */
  double ms_per_step;         /* pbd_autotune: the chosen shape's time per step */
  double default_ms_per_step; /* pbd_autotune: the context's shape before tuning */
} pbd_launch_shape;
int pbd_get_launch_shape(pbd_ctx* ctx, pbd_launch_shape* out);
int pbd_set_launch_shape(pbd_ctx* ctx, const pbd_launch_shape* shape);
/* Time trial_steps graph-launched steps per candidate shape from the context's
 * current state (restored after every trial and at the end, so tuning leaves
 * the state as it found it), coordinate by coordinate, and keep the fastest
 * (a candidate must be 2 % faster than the shape in hand; trial_steps 0: 8).
 * The choice is cached in the process per workload key (particle count to a
 * power of two, grid, variant, phases, scene count) and, when the environment
 * variable PBD_TUNE_CACHE names a file, there too; a cached key is not timed
 * again.  *chosen (may be NULL) receives the shape and both times. */
int pbd_autotune(pbd_ctx* ctx, uint32_t trial_steps, pbd_launch_shape* chosen);

/* Last error message of this context (or, when ctx is NULL, of the last failed
 * pbd_create / pbd_write_frame_arrays / pbd_compute_noalloc of this thread). */
const char* pbd_last_error(pbd_ctx* ctx);

/* ---- One step that allocates nothing ----
 * No counterpart in the reference.  For callers that cannot allocate device
 * memory: code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc.  One call of the step, as pbd_compute makes it (Fluid::compute,
 * Fluid.cu:14-97), on the caller's device arrays of n particles (float4 each,
 * the layout of pbd_buffers), stream-ordered on `stream` (a hipStream_t; NULL
 * is the null stream).  On completion the arrays hold the step's output in its
 * sorted order, as a context's buffers after pbd_compute.  Every call steps as
 * a new context's first compute: the persistent lambdas, delta p and omegas
 * start at zero.  The step's internal buffers are one static device array per
 * GPU (about 11 MiB, held until the process ends), which sets the limits:
 * n <= 32768 and a grid whose Morton cell range holds <= 131072 entries
 * (PBD_ERR_CAPACITY beyond); collisionType 1 is PBD_ERR_UNSUPPORTED.  All calls
 * on one GPU share that array: calls that overlap on one GPU race.  No device
 * allocation, free or memset is made; errors: pbd_last_error(NULL). */
int pbd_compute_noalloc(const pbd_params* p, uint32_t n, float* positions4, float* predicted_positions4,
                        float* velocities4, float* colors4, float* external_forces4, void* stream);

/* ---------------------------------------------------------------------------
 * Batched scenes (no counterpart in the reference, which steps one scene per
 * Fluid::compute, Fluid.cu:14-97).  n scenes share one context and are
 * stepped together: one launch per stage (one graph per substep) for all of
 * them.  Scenes may differ in enclosure (bounds), enclosure damping,
 * relaxation and spawn box; all other parameters must equal scene 0's
 * (PBD_ERR_INVALID otherwise).  Each scene spawns its box at creation; the
 * particle count of a batch is fixed.  Every scene keeps its particles in its
 * own frame (the coordinates of its parameters), so it steps at the FP32
 * resolution of a context of its own.  The kernels see one grid in which scene
 * s occupies a cubic slot; batch frame = scene frame + offset_s
 * (pbd_batch_scene).  Downloads in PBD_FRAME_BATCH add offset_s to positions
 * (an FP32 add on the host). */
typedef struct pbd_batch pbd_batch;
enum { PBD_FRAME_SCENE = 0, PBD_FRAME_BATCH = 1 };
int pbd_batch_create(const pbd_params* scenes, uint32_t n_scenes, pbd_batch** out);
/* frames x substeps substeps of every scene, one graph launch each */
int pbd_batch_step(pbd_batch* b, uint32_t frames);
/* one substep of every scene, launched kernel by kernel */
int pbd_batch_compute(pbd_batch* b);
int pbd_batch_sync(pbd_batch* b);
int pbd_batch_num_scenes(pbd_batch* b, uint32_t* n);
/* particle count, offset (batch frame = scene frame + offset) and the
 * parameters of the scene alone: its own frame, with its slot as the grid
 * (grid_origin, grid_dims = 2^m per axis, grid_cell_size).  A context created
 * with them steps the scene exactly as the batch does; its cell ids are the low
 * 3m bits of the batch's. */
int pbd_batch_scene(pbd_batch* b, uint32_t scene, uint32_t* count, float offset[3], pbd_params* params);
/* per-particle buffer (PBD_BUF_*, not the cell tables) of one scene in sorted
 * order; bytes = count x element size */
int pbd_batch_download(pbd_batch* b, uint32_t scene, int which, int frame, void* dst, size_t bytes);
const char* pbd_batch_last_error(pbd_batch* b);
/* pbd_autotune of the batch's context (all scenes step under one shape). */
int pbd_batch_autotune(pbd_batch* b, uint32_t trial_steps, pbd_launch_shape* chosen);
void pbd_batch_destroy(pbd_batch* b);
/* Free the context (cudaCleanupKernels, kernel/Initialize.h:136-140). */
void pbd_destroy(pbd_ctx* ctx);
/* ABI version (PBD_ABI_VERSION) and the gfx target the kernels were built for. */
int pbd_version(void);
const char* pbd_build_target(void);

#ifdef __cplusplus
}
#endif

#endif /* PBD_PBD_H */
