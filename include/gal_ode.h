/*
 * gal_ode.h -- C ABI of the MI355X batched node-ODE engine.
 *
 * One call evolves a batch of tree-node baryonic ODE systems, each from its
 * own start time to its own end time, with the adaptive Cash-Karp Runge-Kutta
 * (4,5) pair, the scaled error norm and step controller, the driver loop and
 * the node-evolver trial/retry loop of the reference, on one GPU.
 *
 * The reference evolves one node per call through
 *   mergerTreeNodeEvolverStandard%evolve
 *     (source/merger_trees/node_evolver/standard.F90:385-755)
 *   -> odeSolver%solve            (source/numerical/ODE_solver/solver.F90:492-691)
 *   -> gsl_odeiv2_driver2_apply   (source/external/gslODEInitVal2/driver2.c:148-250)
 *   -> gsl_odeiv2_evolve_apply + rkck (GSL 2.6, third party)
 *   -> sc2_control_hadjust        (source/external/gslODEInitVal2/cscal2.c:93-169)
 *   -> RHS callback standardODEs  (source/merger_trees/node_evolver/standard.F90:831-946)
 * and reaches C through the bind(c) interfaces of
 * source/numerical/ODE_solver/solver.F90:62-190.  This header replaces that
 * lower boundary with batched, structure-of-arrays calls.
 *
 * Conventions
 *  - Plain C types only.  Arrays are structure-of-arrays: variable v of node i
 *    is at y[v*ld + i] where ld >= n is the leading dimension.
 *  - "_d" entry points take device pointers (HBM resident, e.g. from
 *    hipMalloc or a torch tensor) and a hipStream_t passed as void*.
 *    "_h" entry points take host pointers; the library stages them.
 *  - Functions return GAL_OK (0) or a negative GAL_E* code; per-node solver
 *    outcomes are reported in status[] with the reference's integer codes.
 *  - No global mutable state: every handle is independent and a handle may be
 *    used from one host thread at a time.
 */
#ifndef GAL_ODE_H
#define GAL_ODE_H

#include <stdint.h>
#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- Library return codes (not per-node statuses) ---------------------- */
#define GAL_OK                 0
#define GAL_E_INVALID         -1   /* bad argument (size, pointer, tolerance) */
#define GAL_E_HIP             -2   /* HIP runtime error                        */
#define GAL_E_NOMEM           -3   /* device allocation failed                 */
#define GAL_E_NODEVICE        -4   /* no usable gfx950 device                  */

/* ---- Per-node statuses: the reference's integer codes ------------------ */
/* GSL_SUCCESS (gsl_errno.h), used by solver.F90:593                          */
#define GAL_STATUS_SUCCESS     0
/* GSL_FAILURE: "step size underflow" (solver.F90:594-607)                    */
#define GAL_STATUS_FAILURE    -1
/* GSL_CONTINUE: post-step changed the state without requiring a reset
   (node_evolver/standard.F90:1180-1183)                                      */
#define GAL_STATUS_CONTINUE   -2
/* odeSolverInterrupt = GSL_EBADFUNC (numerical/ODE_solver/error_codes.F90:33) */
#define GAL_STATUS_INTERRUPT   9
/* errorStatusXCPU (source/error/_module.F90:74)                              */
#define GAL_STATUS_XCPU     1025
/* errorStatusUnderflow = GSL_EUNDRFLW: all trials failed
   (node_evolver/standard.F90:715-718, source/error/_module.F90:72)          */
#define GAL_STATUS_UNDERFLOW  15

/* ---- ODE state layout: component-class order x property order ---------- */
/* Mirrors the serialization order generated by
   python/Galacticus/Build/Components/TreeNodes/ODESolver.py:95-138 for the
   evolvable, non-virtual properties of the standard components
   (source/objects/nodes/components/{hot_halo,disk,spheroid,black_hole}/standard/_class.F90,
    dark_matter_halo/spin/scalar.F90, satellite/standard.F90) with a single
   (metals) abundance slot, plus the hot-halo meta-property added by
   source/nodes/operators/physics/cooling_energy_radiated.F90:120.          */
enum gal_var {
  GAL_V_HOT_MASS = 0,              /* hotHalo%mass                           */
  GAL_V_HOT_ABUNDANCES,            /* hotHalo%abundances (metals)            */
  GAL_V_HOT_ANGULAR_MOMENTUM,      /* hotHalo%angularMomentum                */
  GAL_V_HOT_OUTFLOWED_MASS,        /* hotHalo%outflowedMass                  */
  GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM,
  GAL_V_HOT_OUTFLOWED_ABUNDANCES,
  GAL_V_HOT_UNACCRETED_MASS,
  GAL_V_HOT_UNACCRETED_ABUNDANCES,
  GAL_V_HOT_OUTER_RADIUS,
  GAL_V_HOT_STRIPPED_MASS,
  GAL_V_HOT_STRIPPED_ABUNDANCES,
  GAL_V_HOT_ENERGY_RADIATED,       /* energyRadiatedBensonBower2010          */
  GAL_V_DISK_MASS_STELLAR,         /* disk%massStellar                       */
  GAL_V_DISK_MASS_STELLAR_FORMED,
  GAL_V_DISK_FRACTION_MASS_RETAINED,
  GAL_V_DISK_ABUNDANCES_STELLAR,
  GAL_V_DISK_MASS_GAS,
  GAL_V_DISK_ABUNDANCES_GAS,
  GAL_V_DISK_ANGULAR_MOMENTUM,
  GAL_V_SPHEROID_MASS_STELLAR,     /* spheroid%massStellar                   */
  GAL_V_SPHEROID_MASS_STELLAR_FORMED,
  GAL_V_SPHEROID_ABUNDANCES_STELLAR,
  GAL_V_SPHEROID_MASS_GAS,
  GAL_V_SPHEROID_ABUNDANCES_GAS,
  GAL_V_SPHEROID_ANGULAR_MOMENTUM,
  GAL_V_BH_MASS,                   /* blackHole%mass                         */
  GAL_V_BH_SPIN,
  GAL_V_BH_RADIAL_POSITION,
  GAL_V_SPIN_ANGULAR_MOMENTUM,     /* spin%angularMomentum                   */
  GAL_V_SATELLITE_BOUND_MASS,      /* satellite%boundMass                    */
  GAL_NVAR                         /* = 30                                   */
};

/* ---- Per-node parameters (SoA, GAL_NPARAM_NODE rows) ------------------- */
/* Basic-component quantities that the reference solves analytically
   (nodes/operators/physics/dark_matter_only_mass/interpolate.F90:215-235,
    cosmic_time.F90:81-95) and the spin growth rate set by
   halo_angular_momentum_interpolate.F90.                                    */
enum gal_node_param {
  GAL_NP_TIME_REFERENCE = 0,  /* time at which basic mass == MASS_REFERENCE  */
  GAL_NP_MASS_REFERENCE,      /* halo (basic) mass at TIME_REFERENCE [Msun]  */
  GAL_NP_MASS_RATE,           /* basic%accretionRate [Msun/Gyr]              */
  GAL_NP_SPIN_RATE,           /* d(spin%angularMomentum)/dt [Msun Mpc km/s/Gyr] */
  GAL_NP_IS_SATELLITE,        /* 1.0 for satellites, 0.0 for centrals        */
  GAL_NP_RAM_PRESSURE_FORCE,  /* satellites: ram pressure of the host's hot gas
                                 [Msun Mpc^-3 (km/s)^2], host hot-gas density at
                                 the orbit's pericentre times the squared
                                 pericentric speed (hotHaloRamPressureForce
                                 font2008, hot_halo/ram_pressure_force/Font2008.F90:68-96);
                                 0 for centrals and for no stripping         */
  GAL_NP_HOST_VELOCITY_VIRIAL,/* satellites: virial velocity of the host [km/s]
                                 (hot_halo/ram_pressure_stripping/timescale/
                                 ram_pressure_acceleration.F90:117-132)     */
  GAL_NPARAM_NODE
};

/* ---- Physics parameters (one flat double array, GAL_NPARAM rows) ------- */
/* Names follow the parameter-XML keys of the reference (parameters/quickTest.xml). */
enum gal_param {
  GAL_P_PHYSICS_MODE = 0,           /* 0 standard, 1 box (fixed star-formation timescale and
                                       outflow fractions, no halo gas), 2 test ODEs */
  GAL_P_OMEGA_MATTER,               /* cosmologyParameters/OmegaMatter        */
  GAL_P_OMEGA_DARK_ENERGY,          /* cosmologyParameters/OmegaDarkEnergy    */
  GAL_P_OMEGA_BARYON,               /* cosmologyParameters/OmegaBaryon        */
  GAL_P_HUBBLE_CONSTANT,            /* cosmologyParameters/HubbleConstant     */
  GAL_P_RECYCLED_FRACTION,          /* stellarPopulation/recycledFraction     */
  GAL_P_METAL_YIELD,                /* stellarPopulation/metalYield           */
  GAL_P_SF_DISK_EFFICIENCY,         /* starFormationTimescale(dynamicalTime)/efficiency (disks) */
  GAL_P_SF_DISK_EXPONENT_VELOCITY,
  GAL_P_SF_DISK_TIMESCALE_MINIMUM,
  GAL_P_SF_SPHEROID_EFFICIENCY,     /* same, spheroids                       */
  GAL_P_SF_SPHEROID_EXPONENT_VELOCITY,
  GAL_P_SF_SPHEROID_TIMESCALE_MINIMUM,
  GAL_P_FB_DISK_VELOCITY,           /* stellarFeedbackOutflows(powerLaw)/velocityCharacteristic */
  GAL_P_FB_DISK_EXPONENT,           /* .../exponent                           */
  GAL_P_FB_DISK_TIMESCALE_MINIMUM,  /* rateLimit/timescaleOutflowFractionalMinimum */
  GAL_P_FB_SPHEROID_VELOCITY,
  GAL_P_FB_SPHEROID_EXPONENT,
  GAL_P_FB_SPHEROID_TIMESCALE_MINIMUM,
  GAL_P_REINCORPORATION_MULTIPLIER, /* hotHaloOutflowReincorporation(haloDynamicalTime)/multiplier */
  GAL_P_COOLING_VELOCITY_CUTOFF,    /* coolingRate(whiteFrenk1991)/velocityCutOff */
  GAL_P_CORE_RADIUS_OVER_VIRIAL,    /* hotHaloMassDistributionCoreRadius/coreRadiusOverVirialRadius */
  GAL_P_DEGREES_OF_FREEDOM,         /* coolingTime(simple)/degreesOfFreedom   */
  GAL_P_FRACTION_LOSS_ANGULAR_MOMENTUM, /* coolingInfallTorque(fixed)/fractionLossAngularMomentum */
  GAL_P_RATE_MAXIMUM_EXPULSION,     /* CGMCoolingHeating/rateMaximumExpulsion */
  GAL_P_EFFICIENCY_RADIO_MODE,      /* blackHoleCGMHeating(jetPower)/efficiencyRadioMode */
  GAL_P_BH_ENHANCEMENT_SPHEROID,    /* blackHoleAccretionRate/bondiHoyleAccretionEnhancementSpheroid */
  GAL_P_BH_ENHANCEMENT_HOT_HALO,    /* .../bondiHoyleAccretionEnhancementHotHalo */
  GAL_P_BH_TEMPERATURE_SPHEROID,    /* .../bondiHoyleAccretionTemperatureSpheroid */
  GAL_P_REDSHIFT_REIONIZATION,      /* accretionHalo(simple)/redshiftReionization */
  GAL_P_VELOCITY_SUPPRESSION_REIONIZATION, /* .../velocitySuppressionReionization */
  GAL_P_RADIUS_FACTOR,              /* galacticStructureSolver(fixed)/factor  */
  GAL_P_TOLERANCE_RELATIVE_METALLICITY, /* componentDisk/toleranceRelativeMetallicity */
  GAL_P_BOX_TIMESCALE,              /* starFormationTimescale(fixed)/timescale (box mode) */
  GAL_P_BOX_OUTFLOW_FRACTION,       /* stellarFeedbackOutflows(fixed)/fraction (box mode) */
  GAL_P_OPERATORS,                  /* the optional nodeOperator entries that are listed: GAL_OPERATOR_* bits */
  GAL_P_EXCESS_HEAT_DRIVES_OUTFLOW, /* CGMCoolingHeating/excessHeatDrivesOutflow (1 or 0) */
  GAL_P_BAR_THRESHOLD_STELLAR,      /* galacticDynamicsBarInstability(efstathiou1982)/stabilityThresholdStellar */
  GAL_P_BAR_THRESHOLD_GASEOUS,      /* .../stabilityThresholdGaseous          */
  GAL_P_BAR_TIMESCALE_MINIMUM,      /* .../timescaleMinimum [Gyr]             */
  GAL_P_BAR_J_RETAINED_DISK,        /* .../fractionAngularMomentumRetainedDisk */
  GAL_P_BAR_J_RETAINED_SPHEROID,    /* .../fractionAngularMomentumRetainedSpheroid */
  GAL_P_BH_WIND_EFFICIENCY,         /* blackHoleWind(ciotti2009)/efficiencyWind */
  GAL_P_BH_WIND_SCALES_WITH_RADIATIVE, /* .../efficiencyWindScalesWithEfficiencyRadiative (1 or 0) */
  GAL_P_SPHEROID_ENERGETIC_OUTFLOW, /* componentSpheroid/efficiencyEnergeticOutflow */
  GAL_P_RAM_PRESSURE_FORM_FACTOR,   /* hotHaloRamPressureStripping(font2008)/formFactor */
  GAL_P_BOX_OUTFLOW_FRACTION_SPHEROID, /* stellarFeedbackOutflows(fixed)/fraction of the spheroid (box mode) */
  GAL_P_POST_STEP_ZERO_NEGATIVE_MASSES, /* componentDisk/componentSpheroid postStepZeroNegativeMasses (1 or 0) */
  GAL_NPARAM
};

#define GAL_PHYSICS_STANDARD 0
#define GAL_PHYSICS_BOX      1
#define GAL_PHYSICS_TEST     2

/* Optional node operators (bits of GAL_P_OPERATORS): set when the
   operator appears in the nodeOperator list of the parameter file
   (parameters/quickTest.xml:220-289 lists all four).                        */
#define GAL_OPERATOR_SATELLITE_MASS_LOSS 0x1 /* satelliteMassLoss (satellite/mass_loss/_class.F90:176-200) */
#define GAL_OPERATOR_BAR_INSTABILITY     0x2 /* barInstability (bar_instability.F90:145-248) */
#define GAL_OPERATOR_BLACK_HOLE_WINDS    0x4 /* blackHolesWinds (black_holes/winds.F90:102-133) */
#define GAL_OPERATOR_CGM_OUTER_RADIUS    0x8 /* CGMOuterRadiusRamPressureStripping
                                                (circumgalactic_medium/outer_radius/ram_pressure_stripping.F90:111-242) */

/* ---- Solver flags ------------------------------------------------------ */
#define GAL_FLAG_ENFORCE_NON_NEGATIVITY 0x1  /* enforceNonNegativity (standard.F90:250-256) */
#define GAL_FLAG_REUSE_STEP_SIZE        0x2  /* reuseODEStepSize     (standard.F90:243-249) */
#define GAL_FLAG_SCALES_PROVIDED        0x4  /* use caller scale_abs[] instead of the component scale-set rules */
#define GAL_FLAG_COST_ORDER             0x8  /* claim nodes in decreasing order of a one-RHS stiffness
                                                estimate |t_end-t_start| / sqrt(min_v (|y_v|+s_v)/|dy_v/dt|)
                                                so that the costliest nodes start first (no effect on results) */

/* ---- Cooling-function table ------------------------------------------- */
/* ln(Lambda/[erg cm^3 s^-1]) on a grid uniform in ln T (n_t points from
   ln_t_min with step d_ln_t) and in ln(Z/Zsun) (n_z points).  Storage is
   table[i_z * n_t + i_t].  Follows cieFileInterpolatingFactors /
   cieFileInterpolate (source/cooling/cooling_function/CIE_file.F90:665-735). */
#define GAL_COOLING_NT_MAX 256
#define GAL_COOLING_NZ_MAX  64

typedef struct gal_ode_batch gal_ode_batch;

/* Library and device probing.  Returns GAL_OK when a gfx950 device is usable. */
int gal_ode_version(void);
int gal_ode_device_check(int *n_devices, int *n_cus);

/* Create a handle for batches of up to n_max nodes.  Allocates the device
   buffers it needs for that maximum once. Replaces the per-node
   odeSolverConstructor (solver.F90:335-426) + driver_alloc (driver2.c:31-101). */
int gal_ode_batch_create(int n_max, double tol_abs, double tol_rel, int flags,
                         gal_ode_batch **out);
int gal_ode_batch_destroy(gal_ode_batch *h);

/* Set the GAL_NPARAM physics parameters (host array). */
int gal_ode_batch_set_physics(gal_ode_batch *h, const double *params, int n_params);

/* Upload the cooling table (host arrays). */
int gal_ode_batch_set_cooling_table(gal_ode_batch *h, const double *ln_lambda,
                                    int n_t, double ln_t_min, double d_ln_t,
                                    int n_z, double ln_z_min, double d_ln_z);

/* Launch geometry, validated and kept on the handle: 64 nodes per workgroup
   and 1 to 4 workgroups per CU are admitted.  The integrator has one shape: a
   group of 64 nodes takes four waves and the LDS of a whole CU, and the grid is
   one such group per CU, whatever is set here.  Defaults: 64 and 1. */
int gal_ode_batch_set_launch(gal_ode_batch *h, int nodes_per_block, int blocks_per_cu);

/* Evolve n nodes (device pointers, SoA with leading dimension ld).
 *  y        [GAL_NVAR*ld]  in: state at t_start; out: state at t_end
 *  node_par [GAL_NPARAM_NODE*ld]
 *  t_start, t_end [n]
 *  h_step   [n]  in: node%timeStep() (<=0: none); out: step size to reuse
 *  scale    [GAL_NVAR*ld]  in when GAL_FLAG_SCALES_PROVIDED, else out
 *  status   [n]  per-node status (GAL_STATUS_*)
 *  counters [3*n] or NULL: attempted steps, accepted steps, RHS evaluations
 *  stream   hipStream_t (NULL = default stream)
 * Replaces mergerTreeNodeEvolverStandard%evolve for a wave of nodes
 * (node_evolver/standard.F90:587-740).  Asynchronous on stream.           */
int gal_ode_batch_evolve_d(gal_ode_batch *h, int n, int ld,
                           double *y, const double *node_par,
                           const double *t_start, const double *t_end,
                           double *h_step, double *scale, int *status,
                           int64_t *counters, void *stream);

/* The same evolve in two calls, for callers that run many batches at once on
   several streams.  gal_ode_batch_evolve_d first orders the nodes for
   claiming (a cost estimate per node and a sort, small kernels) and then
   launches the persistent evolve; with several handles on several streams,
   one batch's ordering kernels wait for CUs that other batches' persistent
   launches hold, and its launch starts late.  gal_ode_batch_plan_d runs the
   ordering alone (requires GAL_FLAG_COST_ORDER; reads y, node_par, t_start,
   t_end and, with GAL_FLAG_SCALES_PROVIDED, scale); a later
   gal_ode_batch_evolve_planned_d with the same y pointer, n and ld, and the
   inputs unchanged, launches the evolve in that order.  Results equal
   gal_ode_batch_evolve_d's bit for bit.  A plan serves one evolve; any other
   evolve on the handle discards it; GAL_E_INVALID without a matching plan.
   Asynchronous: enqueue both on one stream, or order their streams.  No
   counterpart in the reference, whose evolver takes one node at a time. */
int gal_ode_batch_plan_d(gal_ode_batch *h, int n, int ld, const double *y,
                         const double *node_par, const double *t_start,
                         const double *t_end, const double *scale,
                         void *stream);
int gal_ode_batch_evolve_planned_d(gal_ode_batch *h, int n, int ld,
                                   double *y, const double *node_par,
                                   const double *t_start, const double *t_end,
                                   double *h_step, double *scale, int *status,
                                   int64_t *counters, void *stream);

/* Host-pointer variant: stages inputs to HBM, evolves, copies results back,
   synchronises.  ld == n.  Used by the Fortran binding. */
int gal_ode_batch_evolve_h(gal_ode_batch *h, int n,
                           double *y, const double *node_par,
                           const double *t_start, const double *t_end,
                           double *h_step, double *scale, int *status,
                           int64_t *counters);

/* Evaluate the RHS dy/dt of n nodes at times t (device pointers, SoA).
   Replaces one call of the standardODEs callback (standard.F90:831-946).  */
int gal_ode_rhs_d(gal_ode_batch *h, int n, int ld, const double *t,
                  const double *y, const double *node_par, double *dydt,
                  void *stream);

/* Apply the scaled step controller to n independent cases (device pointers).
   Case i has dim variables y,yerr,yp,scale at [v*n+i], order ord, step h[i].
   Writes h[i] (adjusted) and result[i] = -1 (DEC), 0 (NIL), +1 (INC), as
   GSL_ODEIV_HADJ_*.  Replaces sc2_control_hadjust (cscal2.c:93-169).     */
int gal_ode_hadjust_d(int n, int dim, int ord, double eps_abs, double eps_rel,
                      double a_y, double a_dydt, const double *y,
                      const double *yerr, const double *yp,
                      const double *scale, const int *is_non_negative,
                      double *h, int *result, void *stream);

/* Allocation-free evolve.  No counterpart in the reference: it is for
   callers that cannot allocate device memory during the call (code under HIP
   graph capture, serving loops, harnesses that forbid hipMalloc).  Same
   arguments and results as creating a handle with tol_abs, tol_rel and flags,
   setting params (host, GAL_NPARAM values) and the cooling table (host), and
   calling gal_ode_batch_evolve_d with the launch shape (64,1), but no handle:
   the parameters, the table and the claim counter live in a static device
   scratch array of the library, one per GPU, of 1 + GAL_NPARAM +
   GAL_COOLING_NT_MAX*GAL_COOLING_NZ_MAX doubles (about 131 KiB), held until the
   process ends.  Tables larger than GAL_COOLING_NT_MAX x GAL_COOLING_NZ_MAX
   are rejected (GAL_E_INVALID).  Nodes are claimed in index order
   (GAL_FLAG_COST_ORDER has no effect; results do not depend on the order).
   Every call on a GPU reuses that GPU's scratch: calls that overlap on one GPU
   (other streams, other host threads) race and must be serialised by the
   caller.  Asynchronous on stream: params and ln_lambda are read by copies
   enqueued on stream, so keep them unchanged until the stream has passed the
   call. */
int gal_ode_evolve_static_d(const double *params, int n_params,
                            const double *ln_lambda, int n_t, double ln_t_min,
                            double d_ln_t, int n_z, double ln_z_min,
                            double d_ln_z, double tol_abs, double tol_rel,
                            int flags, int n, int ld, double *y,
                            const double *node_par, const double *t_start,
                            const double *t_end, double *h_step, double *scale,
                            int *status, int64_t *counters, void *stream);

/* Wall-time limit of each subsequent evolve on this handle, in seconds from
   the start of its launch (<= 0: none).  Checked on the device before every
   Cash-Karp attempt against the GPU's constant-rate realtime counter: a node
   whose attempt would start after the limit returns GAL_STATUS_XCPU (1025)
   with its state and step size as they came in (scales, unless provided,
   are those set at the start of its evolve), as the reference's
   node evolver does when System_Clock passes systemClockMaximum
   (node_evolver/standard.F90:693-705, 860-866); nodes not yet started return
   the same.  The caller converts its own deadline into seconds before each
   call (the Fortran binding does so from systemClockMaximum). */
int gal_ode_batch_set_wall_limit(gal_ode_batch *h, double seconds);

/* Stall limit of the operation-graph executor (gal_tree_evolve_d) on this
   handle, in seconds (<= 0: the default, 60 s): a lane waiting on the graph's
   ready list gives up when no operation at all has become ready for this
   long, and the call then returns GAL_E_HIP with the forest's state
   incomplete.  No counterpart in the reference: it keeps a malformed graph
   from holding the GPU, and a tiny value forces that failure path in tests. */
int gal_ode_batch_set_graph_stall_limit(gal_ode_batch *h, double seconds);

/* Waves per group of 64 nodes, validated and kept on the handle: 1 or 2, the
   default; an evolve with 2 needs one or two workgroups per CU.  The integrator
   uses four waves per group whatever is set here.  No counterpart in the
   reference (launch shape of the GPU kernel). */
int gal_ode_batch_set_rhs_waves(gal_ode_batch *h, int waves);

/* The launch currently set on the handle (by set_launch, set_rhs_waves or
   autotune).  No counterpart in the reference. */
int gal_ode_batch_get_launch(gal_ode_batch *h, int *nodes_per_block, int *blocks_per_cu, int *rhs_waves);

/* Set and return the default launch (64 nodes per workgroup, one workgroup
   per CU, two waves per group): the integrator runs alike at every one, so
   nothing is timed or allocated.  The arguments are those of
   gal_ode_batch_evolve_d and have to describe a batch that it would take;
   scale and status may be NULL. */
int gal_ode_batch_autotune(gal_ode_batch *h, int n, int ld, double *y,
                           const double *node_par, const double *t_start,
                           const double *t_end, double *h_step,
                           double *scale, int *status, void *stream,
                           int *best_nodes_per_block, int *best_blocks_per_cu);

#ifdef __cplusplus
}
#endif
#endif /* GAL_ODE_H */
