/*
 * gamdpy_amd.h -- C ABI of the MI355X (gfx950) per-timestep MD library.
 *
 * The reference (gamdpy) composes numba.cuda device functions into one fused
 * kernel per Simulation; this library replaces that kernel and its launch with
 * hand-written HIP kernels behind the entry points below.  Every signature uses
 * plain C types and host pointers; device memory is owned by the context.
 *
 * Conventions
 *   - every function returns 0 on success and a negative value on failure;
 *     gmd_last_error() then holds a message for the calling thread;
 *   - host arrays are C-contiguous and use the reference's layouts
 *     (positions (N,3) float32, scalars (N,nscalars) float32, ...);
 *   - calls are synchronous on return; one context per host thread.
 */
#ifndef GAMDPY_AMD_H
#define GAMDPY_AMD_H

#ifdef __cplusplus
extern "C" {
#endif

#define GMD_ABI_VERSION 9

typedef struct gmd_ctx gmd_ctx;
typedef struct gmd_rdf gmd_rdf;
typedef struct gmd_batch gmd_batch;
typedef struct gmd_adj gmd_adj;

/* pair function (interactions/potential_functions/): LJ_12_6_sigma_epsilon.py,
 * LJ_12_6.py, make_IPL_n.py, make_LJ_m_n.py, harmonic_repulsion.py, hertzian.py */
enum { GMD_LJ_12_6_SIGMA_EPSILON = 0, GMD_LJ_12_6 = 1, GMD_IPL_N = 2, GMD_LJ_M_N = 3, GMD_HARMONIC_REPULSION = 4,
       GMD_HERTZIAN = 5,
       /* functions read from parameter rows (nparams floats per type pair, the
        * cut last): SAAP.py, and add_potential_functions.py (a sum of two terms) */
       GMD_SAAP = 6, GMD_PAIR_SUM = 7 };
/* cutoff wrapper: none, apply_shifted_potential_cutoff, apply_shifted_force_cutoff */
enum { GMD_CUT_PLAIN = 0, GMD_CUT_SHIFTED_POTENTIAL = 1, GMD_CUT_SHIFTED_FORCE = 2 };
/* compute_plan['nblist'] */
enum { GMD_NBLIST_N_SQUARED = 0, GMD_NBLIST_LINKED_LISTS = 1 };
/* integrators/; NONE = interactions only (tools/Evaluator.py) */
enum { GMD_INTEGRATOR_NONE = 0, GMD_NVE = 1, GMD_NVT = 2, GMD_NVT_LANGEVIN = 3, GMD_NPT_ATOMIC = 4 };
/* misc/make_function.py: constant(value), ramp(value0,x0,value1,x1), sin(period,amplitude,offset) */
enum { GMD_T_CONSTANT = 0, GMD_T_RAMP = 1, GMD_T_SIN = 2 };
/* scalar-saver output columns (fixed order; the host maps them to scalar_names) */
enum { GMD_SAVE_U = 0, GMD_SAVE_W = 1, GMD_SAVE_LAPU = 2, GMD_SAVE_K = 3, GMD_SAVE_FSQ = 4, GMD_SAVE_VOL = 5,
       GMD_SAVE_NCOLS = 6 };

/*
 * Everything Simulation.__init__ (simulation/Simulation.py:73-180) gathers from
 * the Configuration, the PairPotential + NbList, the integrator, the runtime
 * actions and the compute plan.
 */
typedef struct gmd_desc {
    int abi_version;          /* must equal GMD_ABI_VERSION */
    int N, D, ntypes;         /* D must be 3 (the linked-list cell index is 3-D in the reference) */
    float box[3];             /* Orthorhombic lengths */

    /* PairPotential (interactions/pair_potential.py:12-51) */
    int pair_base, cutoff;
    const float *params;      /* ntypes*ntypes*3 float32 (rows of nparams for GMD_SAAP / GMD_PAIR_SUM):
                                 (p0, p1, cut) for [ti][tj]:
                                 LJ_12_6_sigma_epsilon (sigma, epsilon), LJ_12_6 (A12, A6),
                                 IPL_n (A_n, -), LJ_m_n (A_m, A_n),
                                 harmonic_repulsion (epsilon, sigma), hertzian (epsilon, sigma) */
    float pair_exps[2];       /* exponents fixed by the pair function: IPL_n (n, -), LJ_m_n (m, n),
                                 hertzian (alpha, -) (one alpha for all type pairs) */
    float max_cut;            /* max over the cut matrix (pair_potential.py:49) */
    /* GMD_SAAP / GMD_PAIR_SUM: params holds ntypes*ntypes rows of nparams
     * floats (at most 8 parameters, then the cut), and the function is the
     * sum of nterms terms; term k is the pair function term_kind[k] (a
     * GMD_* value 0..6; GMD_HERTZIAN reads eps, alpha, sigma) reading its
     * parameters from term_first[k] on, with exponents term_exps[k] */
    int nparams;
    int nterms;
    int term_kind[2];
    int term_first[2];
    float term_exps[4];

    /* NbList2 / NbListLinkedLists (interactions/nblist.py, nblist_linked_lists.py) */
    int nblist_kind;
    float skin;
    int max_nbs;
    int utilize_niii;         /* compute_plan['UtilizeNIII'] (nblist.py:112-116, pair_potential.py:141-160):
                                 the device keeps the full list (2*max_nbs slots) and forces from it;
                                 each pair's U, W, lapU go to the particle whose half list holds it,
                                 max_nbs bounds that half list, gmd_read_nblist returns it, and the
                                 particles keep the caller's numbering */
    const int *exclusions;    /* N x exclusions_cols, last column = count; NULL = none */
    int exclusions_cols;

    /* integrator */
    int integrator;
    float dt;
    float omega2;             /* NVT.py:148 */
    long long degrees;        /* NVT.py:149 */
    float alpha;              /* NVT_Langevin.py */
    unsigned long long seed;  /* NVT_Langevin.py */
    int tfunc;                /* temperature schedule kind */
    float tparams[4];

    /* compute flags (simulation/get_default_compute_flags.py) */
    int compute_u, compute_w, compute_lap, compute_k, compute_fsq;

    /* column map of the reference scalars array (Configuration.py:109-131) */
    int nscalars, sid_u, sid_w, sid_lap, sid_k, sid_fsq, sid_m;   /* -1 = absent */

    /* runtime actions (runtime_actions/momentum_reset.py, scalar_saver.py) */
    int momentum_reset_every;      /* 0 = off */
    int scalar_save_every;         /* 0 = off */
    int scalar_saves_per_block;

    /* compute plan (simulation/get_default_compute_plan.py) */
    int pb, tp, gridsync;
    int use_graph;                 /* kernel-per-phase path: replay a captured hipGraph */

    /* ConfigurationSaver (runtime_actions/configuration_saver.py:9-148): saves
     * per block (int(log2(steps_per_timeblock)) + 2; 0 = off) of r and r_im at
     * block-local step 0 and at steps 2^b (save index b + 1) */
    int conf_saves_per_block;

    /* Bonds (interactions/bonds.py:12-138) with the harmonic bond function
     * (harmonic_bond_function.py:37-44): nbonds rows (i, j, bond type) of
     * int32 and nbond_types rows (r0, k) of float32; nbonds = 0: no bonds.
     * Each bond adds -dr s to f_i and dr s to f_j (dr = r_j - r_i, minimum
     * image, s = -k (r - r0) / r) and u/2, r^2 s / (2 D), (1 - D) s + k to
     * U, W, lapU of both ends.  The particles keep the caller's numbering. */
    int nbonds;
    const int *bonds;
    int nbond_types;
    const float *bond_params;

    /* NPT_Atomic (integrators/NPT_Atomic.py): integrator = GMD_NPT_ATOMIC,
     * degrees = N D - D, the thermostat and barostat masses of get_params
     * (NPT_Atomic.py:45-56) without their temperature factor, the target
     * temperature in tfunc/tparams and the target pressure in
     * pfunc/pparams.  Needs compute_w.  The box changes every step; with
     * linked lists the cell grid is laid out for a box 5% shorter per side
     * than the starting one, and a run whose box shrinks below that fails. */
    float mass_t, mass_p;
    int pfunc;
    float pparams[4];
} gmd_desc;

typedef struct gmd_device_info {
    int compute_units;
    int wavefront_size;
    int max_threads_per_block;
    long long total_mem;
    char name[64];
    char arch[64];
} gmd_device_info;

/* Library / device ------------------------------------------------------- */
int gmd_abi_version(void);
/* sizeof(gmd_desc) as compiled into the library (binding layout check) */
int gmd_desc_size(void);
const char *gmd_last_error(void);
/* replaces the numba.cuda device queries of get_default_compute_plan.py:24-44 */
int gmd_get_device_info(gmd_device_info *out);

/* Context: replaces Simulation.get_kernels_and_params + make_integrator
 * (Simulation.py:226-347) and the device arrays owned by Configuration,
 * NbList and the integrators. */
int gmd_create(const gmd_desc *desc, gmd_ctx **out);
int gmd_destroy(gmd_ctx *ctx);

/* Configuration.copy_to_device / copy_to_host (Configuration.py:227-243):
 * r, v, f (N,3); scalars (N,nscalars); ptype (N,); r_im (N,3).  NULL = skip. */
int gmd_upload(gmd_ctx *ctx, const float *r, const float *v, const float *f, const float *scalars,
               const int *ptype, const int *r_im);
int gmd_download(gmd_ctx *ctx, float *r, float *v, float *f, float *scalars, int *ptype, int *r_im);

/* Simulation.integrate_self (Simulation.py:271-282): 'steps' integration steps
 * and steps+1 interaction evaluations, starting at time time_zero. */
int gmd_run(gmd_ctx *ctx, float time_zero, int steps);
/* Evaluator.evaluate (tools/Evaluator.py:82-95) on the uploaded state */
int gmd_evaluate(gmd_ctx *ctx);
/* GPU milliseconds of the last gmd_run (hipEvents around the launch) */
int gmd_last_run_ms(gmd_ctx *ctx, float *ms);
/* gmd_run with the steps+1 step kernels launched back to back between two
 * hipEvents: their mean duration (dispatch gaps included); tail_ms is 0
 * (each step's cross-block tail runs inside the next step kernel).  A
 * measurement aid; no counterpart in the reference. */
int gmd_profile_steps(gmd_ctx *ctx, float time_zero, int steps, float *step_ms, float *tail_ms);

/* NbList.d_nbflag (nblist.py:9): [update pending, overflow count, #rebuilds] */
int gmd_read_nbflag(gmd_ctx *ctx, int nbflag[3]);
/* NbList.d_nblist in the reference layout (N, max_nbs+1), count in the last column */
int gmd_read_nblist(gmd_ctx *ctx, int *out);
/* force a rebuild before the next interaction evaluation (nblist.py:67-69 force_update) */
int gmd_force_rebuild(gmd_ctx *ctx);
/* Renumber the particles in cell order at the start of a run once 'steps'
 * steps have passed since the last renumbering (0: never).  Internal only:
 * every host array keeps the caller's order.  Linked-list contexts without
 * exclusions start at 400; no counterpart in the reference. */
int gmd_set_reorder_interval(gmd_ctx *ctx, int steps);
/* Whether the particles are renumbered now (1) or in the caller's order (0),
 * and how many renumberings the context has done.  A diagnostic; no
 * counterpart in the reference. */
int gmd_reorder_stats(gmd_ctx *ctx, int *permuted, long long *renumberings);
/* HBM probe: a plain float4 copy kernel between two fresh device buffers of
 * 'bytes' bytes (a multiple of 16), run 'reps' times after one untimed copy;
 * mean milliseconds per copy.  The known-size workload against which HBM
 * byte counters are scaled (a measurement aid; no counterpart in the
 * reference). */
int gmd_copy_probe(unsigned long long bytes, int reps, float *ms_per_copy);
/* Vector FP32 probe: independent fmaf chains (8 per lane, 'iters' each) over
 * 8 blocks of 256 threads per compute unit; the achieved FP32 TFLOP/s of the
 * code this library is compiled to (no packed FP32).  A measurement aid; no
 * counterpart in the reference. */
int gmd_fma_probe(int iters, float *tflops);

/* NVT.thermostat_state (NVT.py:143): [xi, sum K] */
int gmd_get_thermostat(gmd_ctx *ctx, float state[2]);
int gmd_set_thermostat(gmd_ctx *ctx, const float state[2]);

/* NPT_Atomic.thermostat_state[0], barostat_state[0] and [2] and the box
 * (NPT_Atomic.py:38-39,53; simulation_boxes/orthorhombic.py d_data) between
 * runs: [p_xi/Q, p_eps/W, volume, Lx, Ly, Lz] (the accumulators [1] are zero
 * between steps).  The context must run NPT_Atomic. */
int gmd_get_npt_state(gmd_ctx *ctx, float state[6]);
int gmd_set_npt_state(gmd_ctx *ctx, const float state[6]);

/* ScalarSaver.d_output_array (scalar_saver.py:89-94) of the last block:
 * (scalar_saves_per_block, GMD_SAVE_NCOLS) float32 */
int gmd_read_scalar_output(gmd_ctx *ctx, float *out);

/* ConfigurationSaver.d_conf_array (configuration_saver.py:56-60) of the last
 * block: (conf_saves_per_block, 2, N, 3) float32, [k][0] = r and [k][1] =
 * r_im (as float32) of save k in the caller's numbering; the device array is
 * then cleared, as update_at_end_of_timeblock (configuration_saver.py:84-88)
 * does. */
int gmd_read_conf_output(gmd_ctx *ctx, float *out);

/* Radial distribution (calculators/calculator_radial_distribution.py:76-119).
 * Counts of ordered pairs (ntypes, ntypes, bins) as uint64. */
int gmd_rdf_create(int N, int ntypes, int bins, gmd_rdf **out);
int gmd_rdf_destroy(gmd_rdf *rdf);
/* positions from the context's current device state (no host copy) */
int gmd_rdf_compute_ctx(gmd_rdf *rdf, gmd_ctx *ctx, const int *ptype, unsigned long long *counts);
/* gmd_rdf_compute_ctx in two halves: launch snapshots the context's current
 * positions (on the context's stream) and histograms them on the
 * calculator's own stream, returning at once, so the context's next steps
 * run meanwhile; collect waits for that histogram and returns its counts.
 * One launch at a time per calculator.  The reference's update
 * (calculator_radial_distribution.py:111-119) is the two back to back. */
int gmd_rdf_launch_ctx(gmd_rdf *rdf, gmd_ctx *ctx, const int *ptype);
int gmd_rdf_collect(gmd_rdf *rdf, unsigned long long *counts);
/* positions from a host array (N,3) */
int gmd_rdf_compute_host(gmd_rdf *rdf, const float *r, const int *ptype, const float box[3],
                         unsigned long long *counts);
/* gmd_rdf_compute_host without a calculator object and without any device
 * allocation: no counterpart in the reference.  For callers that cannot
 * allocate device memory (code under graph capture, tight serving loops).
 * Every device buffer (staged positions and types, chunk boxes, thresholds,
 * per-block histograms, counts) lives in one static array of about 11.5 MB
 * per device, held until the process ends.  Limits: N <= 65536,
 * ntypes * ntypes * bins <= 4096; larger sizes are refused with an error.
 * Runs on the null stream and returns when the counts are on the host.  All
 * calls on one device share the array: calls that overlap on one device
 * (other host threads) race. */
int gmd_rdf_compute_host_noalloc(int N, int ntypes, int bins, const float *r, const int *ptype, const float box[3],
                                 unsigned long long *counts);

/* Batches of independent replicas (no counterpart in the reference, which runs
 * one system per Simulation; this replaces running Simulation.run() once per
 * replica).  All replicas share pair function, cutoff, integrator, number of
 * types, tp and pb; N, box, parameters, state point, list kind and runtime
 * actions are per replica.  blocks[r] = blocks that work on replica r (NULL:
 * enough for one particle slot per thread).
 *   GMD_BATCH_PERSISTENT: one cooperative launch per run; the blocks of a
 *     replica meet at their own barrier each step, replicas never wait for
 *     each other;
 *   GMD_BATCH_GRAPH: one launch per step for all replicas, in a hipGraph. */
enum { GMD_BATCH_PERSISTENT = 0, GMD_BATCH_GRAPH = 1 };
int gmd_batch_create(const gmd_desc *descs, int nrep, const int *blocks, int driver, gmd_batch **out);
int gmd_batch_destroy(gmd_batch *batch);
int gmd_batch_size(gmd_batch *batch, int *nrep, int *grid);
/* the context of replica rep, for gmd_upload/gmd_download/gmd_read_* and the
 * RDF; gmd_run, gmd_evaluate and gmd_destroy refuse it */
int gmd_batch_context(gmd_batch *batch, int rep, gmd_ctx **out);
/* 'steps' steps of every replica (Simulation.integrate_self per replica) */
int gmd_batch_run(gmd_batch *batch, float time_zero, int steps);
/* Bring the state of every replica to the host in one go: the next
 * gmd_download of each replica (before it is run or uploaded again) only
 * copies it. */
int gmd_batch_fetch(gmd_batch *b);
int gmd_batch_last_run_ms(gmd_batch *batch, float *ms);

/* Differentiable NVE trajectory (no counterpart in the reference; it adds
 * gradients of a trajectory observable with respect to the LJ parameters and
 * the initial positions, for fitting potentials to structural data).
 * Model: LJ_12_6_sigma_epsilon with gamdpy's shifted-force cutoff
 * (apply_shifted_force_cutoff.py:29-37, s(r) - s(rc)) at a fixed cut;
 * NVE leap-frog (NVE.py:59-105); float32 forward.  The adjoint pass reads the
 * positions of every step, which stay in device memory up to 4 GiB (16 bytes a
 * particle and step) where there is room for them, or recomputes them from
 * checkpoints every ckpt_every steps.
 * Observable: H[c][k] = sum over frames (every rdf_every steps, including 0
 * and, when it is a multiple, nsteps) and unordered pairs of class c of
 * max(0, exp(-(d - r_k)^2 / (2 w^2)) - exp(-12.5)) for |d - r_k| < 5 w,
 * r_k = (k + 1/2) rdf_rmax / rdf_bins, w = rdf_width; classes enumerate
 * type pairs a <= b in row order. */
typedef struct gmd_adj_desc {
    int N, ntypes;
    float box[3];
    float dt;
    int nsteps, ckpt_every;
    int rdf_every, rdf_bins;
    float rdf_rmax, rdf_width;
} gmd_adj_desc;
int gmd_adj_create(const gmd_adj_desc *desc, const int *ptype, const float *mass, gmd_adj **out);
int gmd_adj_destroy(gmd_adj *adj);
/* params: ntypes*ntypes*3 float32 (sigma, epsilon, cut), symmetric; r0, v0 (N,3);
 * H: nclass*bins float64; r_end, v_end (N,3) or NULL.  Replaces what the last
 * forward pass left for gmd_adj_backward, also when it fails. */
int gmd_adj_forward(gmd_adj *adj, const float *params, const float *r0, const float *v0, double *H, float *r_end,
                    float *v_end);
/* dLdH: nclass*bins; grad_params: nclass*2 float64 (dL/dsigma, dL/depsilon per
 * class); grad_r0, grad_v0 (N,3) (grad_v0 may be NULL) */
int gmd_adj_backward(gmd_adj *adj, const double *dLdH, double *grad_params, float *grad_r0, float *grad_v0);
int gmd_adj_last_ms(gmd_adj *adj, float *fwd_ms, float *bwd_ms);
/* keep checkpoints only, as a trajectory of more than 4 GiB does, and recompute
 * between them in the backward pass (same results; a forward pass before the
 * call is dropped).  Where they find no memory: an error, and the handle keeps
 * the trajectory. */
int gmd_adj_use_checkpoints(gmd_adj *adj);

#ifdef __cplusplus
}
#endif
#endif /* GAMDPY_AMD_H */
