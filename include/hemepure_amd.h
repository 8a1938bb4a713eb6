/*
 * hemepure_amd.h -- C ABI of the MI355X D3Q19 collide-and-stream library.
 *
 * The reference (HemePure) has no foreign-function interface: its hot path is a
 * set of compile-time CRTP templates driven by lb::LBM<D3Q19>.  Every entry
 * point below replaces one call of that host API; the comment on each names the
 * reference interface (paths relative to the HemePure source tree).  All entry
 * points return 0 on success and a negative HLB_E* code on failure;
 * hlb_last_error() returns the message of the calling thread's last failure.
 * No torch or HIP types appear in the signatures: plain pointers and sizes.
 *
 * Threading: a handle is single-threaded, like the reference's LBM object
 * (one thread per MPI rank).  Work is ordered on the handle's HIP stream.
 */
#ifndef HEMEPURE_AMD_H
#define HEMEPURE_AMD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- status codes ------------------------------------------------------ */
#define HLB_OK 0
#define HLB_EINVAL -1    /* bad argument or configuration */
#define HLB_EGEOMETRY -2 /* geometry the pull scheme cannot represent */
#define HLB_EDEVICE -3   /* HIP runtime failure */
#define HLB_ERANGE -4    /* e.g. iolet site outside a parabolic radius */

/* ---- enums mirroring the reference's build-time selections ------------- */
/* Link intersection type, GeometrySiteLink::IntersectionType
 * (src/geometry/GeometrySiteLink.h). */
#define HLB_LINK_NONE 0
#define HLB_LINK_WALL 1
#define HLB_LINK_INLET 2
#define HLB_LINK_OUTLET 3

/* HEMELB_KERNEL (src/CMakeLists.txt:47-48, src/lb/BuildSystemInterface.h:24-60). */
#define HLB_KERNEL_LBGK 0
#define HLB_KERNEL_TRT 1
#define HLB_KERNEL_LES 2 /* LBGKLESSL: Smagorinsky (C_s = 0.1), sponge layer by hlb_set_sponge */

/* HEMELB_WALL_BOUNDARY (src/lb/BuildSystemInterface.h:165-197). */
#define HLB_WALL_SBB 0
#define HLB_WALL_BFL 1
#define HLB_WALL_GZS 2 /* GuoZhengShiDelegate (LBGK and TRT) */

/* HEMELB_{INLET,OUTLET}_BOUNDARY and their wall-corner variants
 * (src/lb/BuildSystemInterface.h:215-331): Nash pressure or Ladd velocity. */
#define HLB_IOLET_NASH 0
#define HLB_IOLET_LADD 1

/* Iolet value providers (src/lb/iolets/). */
#define HLB_IOLET_COSINE 0    /* InOutLetCosine */
#define HLB_IOLET_PARABOLIC 1 /* InOutLetParabolicVelocity */
#define HLB_IOLET_FILEVEL 2   /* InOutLetFileVelocity, table already in lattice units */
#define HLB_IOLET_WK2 3       /* InOutLetWK2 */
#define HLB_IOLET_WK3 4       /* InOutLetWK3 */
#define HLB_IOLET_FILEPRES 5  /* InOutLetFile: density per 0-indexed step (hlb_iolet_file_table) */
#define HLB_IOLET_WOMERSLEY 6 /* InOutLetWomersleyVelocity */

/* Storage precision of the distributions. */
#define HLB_FP64 0
#define HLB_FP32_SHIFTED 1

/* Order of the slabs (x layers of occupied 8^3 tiles) in device memory and in
 * the launch.  TILE: tile after tile (z fastest), each tile's layers in turn.
 * LAYER: layer 0 of every tile, then layer 1, ...; with the XCD-contiguous
 * launch order each XCD then walks one layer, and a slab's y neighbours,
 * which share the cache lines of its face lanes, come within its L2 window.
 * AUTO (0): LAYER when the median distance from a slab to its y neighbour in
 * TILE order exceeds that window (431 slabs), else TILE; lattices whose
 * distributions take 64 to 256 MB and run along y or z enumerate their tiles in
 * sections of 8 tiles along that axis first.  No effect on
 * results; hlb_get_params reports the order chosen. */
#define HLB_ORDER_AUTO 0
#define HLB_ORDER_TILE 1
#define HLB_ORDER_LAYER 2

/* hlb_step flags */
#define HLB_STEP_PROPERTIES 1u /* fill rho, u and WSS during the last step */

/* ---- geometry (the content of a .gmy file, decoded) --------------------- */
/* One record per fluid site, in any order.  Directions are D3Q19 1..18
 * (src/lb/lattices/D3Q19.cc:15-17).  Mirrors GeometrySite/GeometrySiteLink
 * (src/geometry/GeometrySite.h, GeometrySiteLink.h) as produced by
 * GeometryReader::ParseSite (src/geometry/GeometryReader.cc:851-935). */
typedef struct hlb_geometry {
  int32_t blocks[3];          /* block counts; the site grid is blocks*block_size */
  int32_t block_size;         /* 8 in every .gmy file */
  int64_t n_sites;
  const int32_t* coords;      /* n*3 global site coordinates */
  const uint8_t* link_type;   /* n*18 HLB_LINK_* */
  const int32_t* link_iolet;  /* n*18 iolet id (-1 if none) */
  const float* link_dist;     /* n*18 fraction of the link before the intersection */
  const uint8_t* normal_avail;/* n */
  const float* normal;        /* n*3 wall normal as stored (un-normalised) */
} hlb_geometry;

/* One inlet or outlet: position/normal/radius from the XML plus the
 * provider's parameters (src/configuration/SimConfig.cc:268-400, 725-830). */
typedef struct hlb_iolet_desc {
  int32_t kind;            /* HLB_IOLET_COSINE .. HLB_IOLET_WOMERSLEY */
  int32_t warmup;          /* cosine / parabolic warm-up steps */
  double position[3];      /* lattice units */
  double normal[3];        /* normalised in double, as InOutLet::SetNormal */
  double radius;           /* velocity and Windkessel iolets */
  double density_mean;     /* cosine */
  double density_amp;      /* cosine */
  double phase;            /* cosine, radians */
  double period;           /* cosine, Womersley: lattice steps */
  double max_speed;        /* parabolic */
  const double* table;     /* file velocity: max speed per 1-indexed step;
                              file pressure: density per 0-indexed step */
  int64_t table_len;
  double density_min;      /* file pressure: GetDensityMin */
  double pressure_gradient_amplitude; /* Womersley, lattice units */
  double womersley_number;            /* Womersley */
  double area;             /* Windkessel */
  double resistance;       /* WK2 */
  double r_c;              /* WK3 characteristic resistance */
  double r_p;              /* WK3 peripheral resistance */
  double capacitance;      /* WK2 / WK3 */
} hlb_iolet_desc;

/* Collision and boundary selection plus LbmParameters
 * (src/lb/LbmParameters.h:29-45; relaxation_parameter SimConfig.cc:165-169). */
typedef struct hlb_params {
  int32_t kernel;     /* HLB_KERNEL_* */
  int32_t wall_bc;    /* HLB_WALL_* */
  int32_t inlet_bc;   /* HLB_IOLET_NASH / HLB_IOLET_LADD */
  int32_t outlet_bc;
  int32_t precision;  /* HLB_FP64 */
  int32_t slab_order; /* HLB_ORDER_*: read by hlb_create; fixed afterwards */
  double tau;
  double trt_lambda;
} hlb_params;

typedef struct hlb_lattice* hlb_handle;

/* ---- errors ------------------------------------------------------------- */
/* Replaces hemelb::Exception messages (src/Exception.h:25) and the
 * std::exit(16) of InOutLetParabolicVelocity.cc:39-45. */
const char* hlb_last_error(void);

/* ---- lifecycle ---------------------------------------------------------- */
/* Builds the lattice and uploads it to the current HIP device.  Replaces
 * LatticeData::LatticeData -> ProcessReadSites + InitialiseNeighbourLookups
 * (src/geometry/LatticeData.cc:69-517), LBM::LBM + ReadParameters
 * (src/lb/lb.hpp:361-374), BoundaryValues::BoundaryValues
 * (src/lb/iolets/BoundaryValues.cc:20-81) and LBM::InitCollisions
 * (src/lb/lb.hpp:73-117).  Fails with HLB_EGEOMETRY when a link's type
 * disagrees with its neighbour's fluidity (two or zero writers of one
 * distribution in the reference's push step). */
int hlb_create(const hlb_geometry* geom, const hlb_params* params, const hlb_iolet_desc* inlets,
               int n_inlets, const hlb_iolet_desc* outlets, int n_outlets, hlb_handle* out);
/* With params == NULL hlb_create builds only the lattice tables (the
 * reference's LatticeData before an LBM exists); the collision/boundary
 * selection and the iolets then come from hlb_set_params and hlb_set_iolets.
 * hlb_set_params replaces LBM::ReadParameters / LbmParameters::Update
 * (src/lb/lb.hpp:361-374, src/lb/LbmParameters.h:40-44): once the lattice has
 * a device state only tau and trt_lambda may change.  hlb_set_iolets replaces
 * BoundaryValues::BoundaryValues (src/lb/iolets/BoundaryValues.cc:20-81) and
 * is allowed until the lattice has a device state. */
int hlb_set_params(hlb_handle h, const hlb_params* params);

/* The sponge layer of the LES kernel (LBGKLESSpongeLayer,
 * src/lb/kernels/LBGKLESSpongeLayer.h:87-148; its parameters are
 * LbmParameters::ViscosityRatio, SpongeLayerWidth and SpongeLayerLifetime,
 * src/lb/LbmParameters.h:84-86, read from <sponge_layer> at
 * src/configuration/SimConfig.cc:705-722).  Every site within `width`
 * (lattice units) of an outlet position gets a raised relaxation time vTau;
 * up to half the lifetime a site relaxes with vTau (the Smagorinsky time
 * where vTau equals tau), then linearly into the Smagorinsky time, which
 * alone applies from step `lifetime` on.  Lifetime 0 (the default) is pure
 * Smagorinsky LES.  HLB_EINVAL for another kernel, a width <= 0 or a
 * non-finite ratio.  Recomputed after hlb_set_params / hlb_set_iolets. */
int hlb_set_sponge(hlb_handle h, double viscosity_ratio, double width, int64_t lifetime);
int hlb_get_params(hlb_handle h, hlb_params* out);
int hlb_set_iolets(hlb_handle h, const hlb_iolet_desc* inlets, int n_inlets, const hlb_iolet_desc* outlets,
                   int n_outlets);
/* Replaces LBM::~LBM / LatticeData::~LatticeData. */
void hlb_destroy(hlb_handle h);

/* ---- initial conditions ------------------------------------------------- */
/* EquilibriumInitialCondition::SetFs (src/lb/InitialCondition.hpp:30-43):
 * f = f_eq(rho0, 0) at every site; the step counter restarts at t0 (1 =
 * SimulationState's start, src/lb/SimulationState.cc:17). */
int hlb_init_equilibrium(hlb_handle h, double rho0, int64_t t0);
/* CheckpointInitialCondition::SetFs (src/lb/InitialCondition.hpp:46-50,
 * LocalDistributionInput::LoadDistribution): pre-collision f in the
 * reference's contiguous site order, AoS f[site*19+d], double. */
int hlb_upload_f(hlb_handle h, const double* f, int64_t t0);

/* ---- the hot path ------------------------------------------------------- */
/* Advances nsteps time steps, each one the reference's
 * LBM::RequestComms/PreSend/PreReceive/PostReceive/EndIteration sequence
 * (src/lb/lb.hpp:192-347) plus the BoundaryValues comms of its iolets, as
 * fused pull-scheme collide+stream launches on the handle's stream.
 * HLB_STEP_PROPERTIES fills density, velocity and wall-shear-stress caches
 * during the last step (BaseStreamer::UpdateMinsAndMaxes,
 * src/lb/streamers/BaseStreamer.h:88-120).  Asynchronous. */
int hlb_step(hlb_handle h, int64_t nsteps, uint32_t flags);
/* Launch variant of the steady-state step, 0..35 = shape + 6 * level: shape
 * 0..5 = workgroups of 128/256/64 slots without/with the XCD-contiguous
 * order, level 0..3 = at most (unlimited, 4, 3, 2) waves per SIMD, level
 * 4..5 = compiled for at least (5, 6) waves per SIMD in FP64 and (6, 7) in
 * the FP32-shifted form.  Until a variant is set or autotuned a lattice (and
 * a batch) reports variant 1, or its non-temporal-store twin (FP64 55, FP32
 * 109) while its distributions exceed the 256 MB Infinity Cache, and is
 * launched in the shape that fits their size: variant 5 while they fit the
 * cache, 55 / 109 up to 2.5 times its size (a batch 182), 92 / 182 beyond.
 * Setting the reported variant launches that variant itself.  FP32 lattices with
 * wall or iolet links between two fluid sites, and batches that hold one, are
 * launched in variant 5's shape with the set or default one's store policy.
 * FP64 36..53 = block + 3 * level with
 * block 0..2 = 128/256/64 slots in the XCD-chunk order (chunks of 32
 * workgroup tiles dealt to the XCDs in turn).  The FP32-shifted form takes
 * 0..35, 36..71 = 0..35 with two consecutive slabs per wavefront (both
 * slabs' loads in flight together), 72..89 = the XCD-chunk shapes and
 * 90..107 = those with two slabs per wavefront.  FP64 54..107 and FP32
 * 108..215 repeat 0..53 / 0..107 with the post-collision row written by
 * non-temporal stores (faster where the arrays are far larger than the
 * caches, slower where they fit the Infinity Cache).
 * No counterpart in the reference.  hlb_autotune times every variant over
 * trial_steps real steps of the lattice (they advance it; replayed where the
 * lattice's long sequences are) and keeps the fastest; results do not depend on
 * the variant. */
int hlb_set_variant(hlb_handle h, int variant);
int hlb_variant(hlb_handle h);
int hlb_autotune(hlb_handle h, int64_t trial_steps, int* variant, double* ms_per_step);
/* Like hlb_step, timing the launches with HIP events recorded on the handle's
 * stream; blocks until done and returns the elapsed milliseconds.  A
 * sequence that hlb_step would replay (hlb_set_graphs) and that was not seen
 * before is captured ahead of the first event, so the timed region holds the
 * replay only; any other is launched step by step within it. */
int hlb_step_timed(hlb_handle h, int64_t nsteps, uint32_t flags, double* ms);
/* No counterpart in the reference (its steps are host loops over site
 * ranges).  Step sequences (16 to 1024 steps) of small lattices are captured
 * into HIP graphs on first use and replayed (the default, enable = 1), so they
 * are not bound by per-launch cost; short sequences and lattices whose steps
 * hide it, and with enable = 0 every sequence, are launched step by step.
 * Results are bit-identical either way.  Changing it, or tau via hlb_set_params,
 * drops the captured graphs. */
int hlb_set_graphs(hlb_handle h, int enable);
/* Captured sequences the handle holds (at most 8), -1 for a null handle. */
int hlb_captured_graphs(hlb_handle h);
/* Blocks until the handle's stream is idle. */
int hlb_synchronize(hlb_handle h);

/* ---- extraction / checkpoint ------------------------------------------- */
/* LatticeData::GetFOld after LBM::EndIteration's swap (src/lb/lb.hpp:336-346):
 * the pre-collision f entering step hlb_timestep(h), AoS f[site*19+d] in the
 * reference's site order. */
int hlb_download_f(hlb_handle h, double* f);
/* MacroscopicPropertyCache density/velocity/WSS of the last step run with
 * HLB_STEP_PROPERTIES (src/lb/MacroscopicPropertyCache.h:24-106).  u is n*3;
 * WSS is DBL_MAX (NO_VALUE) at sites without a wall link.  Any may be NULL. */
int hlb_get_fields(hlb_handle h, double* rho, double* u, double* wss);
/* The stress caches of MacroscopicPropertyCache (src/lb/MacroscopicPropertyCache.h)
 * that step T's collision fills (BaseStreamer::UpdateMinsAndMaxes,
 * src/lb/streamers/BaseStreamer.h:120-220), computed on the device from the
 * state entering step T = hlb_timestep(h), lattice units, site order:
 * tensor n*6 (full stress tensor xx, xy, xz, yy, yz, zz: -Pi - (rho-1)Cs2 I,
 * Lattice.h:1096-1111), von Mises stress n (:983-1001), shear rate n
 * (:1159-1180), and n*3 each the traction, its tangential and its normal
 * projection at wall sites (:1017-1079; zero vectors elsewhere).  Any may be
 * NULL. */
int hlb_get_stress(hlb_handle h, double* tensor, double* von_mises, double* shear_rate, double* traction,
                   double* tangential, double* normal);
/* The same as one n*17 record array: per site the tensor's 6, von Mises, shear
 * rate, traction 3, tangential 3, normal 3. */
int hlb_get_stress_rows(hlb_handle h, double* rows);
/* SimulationState::GetTimeStep (src/lb/SimulationState.cc:50): the 1-indexed
 * step that runs next. */
int64_t hlb_timestep(hlb_handle h);
/* StabilityTester (src/lb/StabilityTester.h:100-117): 1 if every
 * distribution entering the next step is > 0 (and not NaN). */
int hlb_stability(hlb_handle h, int* stable);

/* ---- property extraction files (.xtr + .off) ---------------------------- */
/* Field types, numbered as OutputField::FieldType (src/extraction/
 * OutputField.h:17-31).  A field is
 * written under its given name, or its type name ("pressure", "velocity",
 * "shearstress", "distributions", "mpirank") when none is given, as
 * SimConfig::DoIOForPropertyField (SimConfig.cc:565-580) defaults it.
 * Wall extension has no source here (only the elastic GZS wall sets it) and
 * is written as 0. */
#define HLB_FIELD_PRESSURE 0                       /* mmHg, offset REFERENCE_PRESSURE_mmHg */
#define HLB_FIELD_VELOCITY 1                       /* m/s, 3 floats */
#define HLB_FIELD_SHEAR_STRESS 2                   /* Pa, wall sites; elsewhere inf */
#define HLB_FIELD_VON_MISES_STRESS 3               /* Pa */
#define HLB_FIELD_SHEAR_RATE 4                     /* 1/s */
#define HLB_FIELD_STRESS_TENSOR 5                  /* Pa, xx xy xz yy yz zz */
#define HLB_FIELD_TRACTION 6                       /* Pa, 3 floats; NaN where no normal */
#define HLB_FIELD_TANGENTIAL_PROJECTION_TRACTION 7 /* Pa, 3 floats */
#define HLB_FIELD_NORMAL_PROJECTION_TRACTION 8     /* Pa, 3 floats */
#define HLB_FIELD_WALL_EXTENSION 9                 /* m; 0 (no elastic walls) */
#define HLB_FIELD_DISTRIBUTIONS 10                 /* 19 floats, lattice units */
#define HLB_FIELD_MPI_RANK 11                      /* 0: one process */
/* Geometry selectors (the src/extraction/...Selector.cc classes). */
#define HLB_SELECT_WHOLE 0
#define HLB_SELECT_SURFACE 1 /* wall sites */
#define HLB_SELECT_INLET 2   /* SiteType INLET_TYPE */
#define HLB_SELECT_OUTLET 3  /* SiteType OUTLET_TYPE */
#define HLB_SELECT_PLANE 4   /* |distance| <= voxel/2, within radius if > 0 */
#define HLB_SELECT_SPHERE 5  /* within radius of point */
#define HLB_SELECT_LINE 6    /* within voxel/sqrt2 of the segment point..point2 */
#define HLB_SELECT_SURFACE_POINT 7  /* wall sites within sqrt3 voxels of point */
#define HLB_SELECT_SURFACE_SPHERE 8 /* wall sites within radius of point */
/* One <propertyoutput> of the XML (SimConfig::DoIOForPropertyOutputFile,
 * src/configuration/SimConfig.cc:420-560): the fields, the
 * selector with its point (m), normal and radius (m), and the unit
 * conversion (voxel size in m, time step in s, origin in m). */
typedef struct hlb_xtr_spec {
  const int32_t* fields;
  const char* const* names; /* n_fields names, or NULL; a NULL entry: type name */
  int32_t n_fields;
  int32_t selector;
  double voxel_size;
  double time_step;
  double origin[3];
  double point[3];
  double normal[3];
  double radius;
  double point2[3]; /* the line's second end */
} hlb_xtr_spec;
typedef struct hlb_xtr* hlb_xtr_handle;
/* LocalPropertyOutput::LocalPropertyOutput (src/extraction/
 * LocalPropertyOutput.cc:27-198): selects the sites, creates the file (it
 * must not exist) and writes the headers; with a distributions field also the
 * .off file (WriteOffsetFile, :331-357). */
int hlb_xtr_open(hlb_handle h, const char* path, const hlb_xtr_spec* spec, hlb_xtr_handle* out);
/* Record T holds what the reference writes at the end of step T
 * (PropertyActor::EndIteration, src/extraction/PropertyActor.cc:94-99): the
 * distributions that entered step T and step T's property caches.  Call
 * hlb_xtr_capture before step T (it copies f and computes the stress caches
 * when a field needs them), run
 * step T with HLB_STEP_PROPERTIES, then hlb_xtr_write (LocalPropertyOutput::
 * Write, :216-327), which returns T.  A distributions-only record needs no
 * step in between. */
int hlb_xtr_capture(hlb_xtr_handle x);
int hlb_xtr_write(hlb_xtr_handle x, int64_t* timestep);
/* Writes one record from caller arrays in the lattice's site order, lattice
 * units: rho n, u n*3, wss n, f n*19, stress n*17 (per site the stress
 * tensor's 6, von Mises, shear rate, traction 3, tangential 3, normal 3, as
 * hlb_get_stress_rows returns them); arrays no field uses may be NULL. */
int hlb_xtr_write_fields(hlb_xtr_handle x, int64_t timestep, const double* rho, const double* u,
                         const double* wss, const double* f, const double* stress);
int64_t hlb_xtr_site_count(hlb_xtr_handle x);
void hlb_xtr_close(hlb_xtr_handle x);
/* LocalDistributionInput::LoadDistribution (src/extraction/
 * LocalDistributionInput.cc:48-177): reads the record of timestep `target`
 * (the last record when target < 0) of a distributions-only .xtr and its .off
 * file, checks every site's coordinates against the lattice, and returns the
 * timestep and f (n*19, float values widened).  Pass both to hlb_upload_f to
 * restart: CheckpointInitialCondition (src/lb/InitialCondition.hpp:46-50,
 * InitialCondition.cc:18-21) sets the next step to the record's. */
int hlb_checkpoint_read(hlb_handle h, const char* path, int64_t target, int64_t* timestep, double* f);

/* ---- batches of FP32-shifted lattices ----------------------------------- */
/* No counterpart in the reference, which runs one lattice per process: the
 * ensemble and serving forms advance many independent lattices (members,
 * each created with hlb_create and HLB_FP32_SHIFTED and given an initial
 * condition) with one step launch per time step over all of them.  Members
 * stay owned by the caller, keep their own step counter and iolet state, and
 * compute exactly what they compute alone.  A member may join or leave
 * between calls; destroying a member removes it.  hlb_step on a member and
 * batch steps are ordered. */
typedef struct hlb_batch* hlb_batch_handle;
int hlb_batch_create(hlb_batch_handle* out);
void hlb_batch_destroy(hlb_batch_handle b);
int hlb_batch_add(hlb_batch_handle b, hlb_handle member);
int hlb_batch_remove(hlb_batch_handle b, hlb_handle member);
int hlb_batch_size(hlb_batch_handle b);
int64_t hlb_batch_sites(hlb_batch_handle b);
/* Advances every member by nsteps (HLB_STEP_PROPERTIES: fields of the last
 * step).  Asynchronous with respect to the host. */
int hlb_batch_step(hlb_batch_handle b, int64_t nsteps, uint32_t flags);
/* Like hlb_batch_step for at most 1024 steps; blocks and returns the device
 * milliseconds of the launches (HIP events on the batch's stream). */
int hlb_batch_step_timed(hlb_batch_handle b, int64_t nsteps, uint32_t flags, double* ms);
/* As hlb_set_graphs, for the batch's sequences (default on). */
int hlb_batch_set_graphs(hlb_batch_handle b, int enable);
int hlb_batch_captured_graphs(hlb_batch_handle b);
/* Launch variant, as for hlb_set_variant of an FP32-shifted lattice (0..215). */
int hlb_batch_set_variant(hlb_batch_handle b, int variant);
int hlb_batch_variant(hlb_batch_handle b);
/* Times each launch variant over trial_steps real steps of every member and
 * keeps the fastest. */
int hlb_batch_autotune(hlb_batch_handle b, int64_t trial_steps, int* variant, double* ms_per_step);

/* ---- serving: a solve-request loop over one batch ------------------------ */
/* No counterpart in the reference.  Requests are submitted at any time, from
 * any thread (hlb_server_submit builds the tables on the calling thread), and
 * run in the FP32-shifted form; each hlb_server_advance admits queued
 * requests in arrival order while their device bytes fit the budget (a
 * request that does not fit is passed over by later ones that do, at most 8
 * times, then admission waits for it), advances all running requests by one
 * quantum in one batch, measures the cycle-to-cycle max |du| of requests at
 * a cycle end, and retires requests that converged (max |du| < tolerance) or
 * reached max_steps, keeping their rho, u and WSS on the host.  Times are
 * seconds since hlb_server_create.  hlb_server_advance is called from one
 * thread at a time.  Both modes step in the default launch shape for the size of
 * the running distributions (see hlb_set_variant).
 * HLB_SERVE_PLAIN (hlb_server_set_mode, before the first submission) serves
 * the way the reference runs many cases: one request at a time in arrival
 * order, each stepped alone with hlb_step, in either storage form -- the
 * one-at-a-time baseline for the same arrivals. */
#define HLB_SERVE_BATCHED 0
#define HLB_SERVE_PLAIN 1
#define HLB_REQ_QUEUED 0
#define HLB_REQ_RUNNING 1
#define HLB_REQ_CONVERGED 2
#define HLB_REQ_DONE 3   /* reached max_steps without converging */
#define HLB_REQ_FAILED 4

typedef struct hlb_request {
  const hlb_geometry* geom;
  hlb_params params;            /* batched mode: precision must be HLB_FP32_SHIFTED */
  const hlb_iolet_desc* inlets;
  int32_t n_inlets;
  int32_t pad0_;
  const hlb_iolet_desc* outlets;
  int32_t n_outlets;
  int32_t pad1_;
  int64_t max_steps;            /* cap, rounded up to the quantum */
  int64_t period;               /* steps per cycle of the convergence test (multiple of the quantum) */
  double tolerance;             /* cycle-to-cycle max |du|; 0 runs max_steps */
  double rho0;                  /* initial equilibrium density */
} hlb_request;

typedef struct hlb_request_status {
  int32_t state;                /* HLB_REQ_* */
  int32_t cycles;
  int64_t steps;
  int64_t sites;
  int64_t device_bytes;
  double delta;                 /* last cycle-to-cycle max |du| (inf before two cycle ends) */
  double t_submit, t_admit, t_done;
} hlb_request_status;

typedef struct hlb_server* hlb_server_handle;
int hlb_server_create(int64_t budget_bytes, int64_t quantum_steps, hlb_server_handle* out);
void hlb_server_destroy(hlb_server_handle s);
int hlb_server_set_mode(hlb_server_handle s, int mode);
/* Builds the request's lattice tables on the host and queues it. */
int hlb_server_submit(hlb_server_handle s, const hlb_request* r, int64_t* id);
int hlb_server_advance(hlb_server_handle s, int* running, int* queued);
int hlb_server_status(hlb_server_handle s, int64_t id, hlb_request_status* out);
/* Fields of a finished request, reference site order. */
int hlb_server_fields(hlb_server_handle s, int64_t id, double* rho, double* u, double* wss);
int hlb_server_release(hlb_server_handle s, int64_t id);
int64_t hlb_server_site_steps(hlb_server_handle s);
int64_t hlb_server_bytes_in_use(hlb_server_handle s);
/* Device bytes a lattice holds once it has a state (admission accounting). */
int64_t hlb_device_bytes(hlb_handle h);

/* Monitors from the fields of the last step run with HLB_STEP_PROPERTIES,
 * reduced on the device over the fluid sites: out[0] smallest density,
 * out[1] largest density, out[2] largest |u| (the DensityTracker of
 * IncompressibilityChecker, src/lb/IncompressibilityChecker.hpp:170-195;
 * max relative density difference = (out[1] - out[0]) / 1), out[3] total
 * mass sum rho in FP64, summed in a fixed order (reproducible). */
int hlb_monitor(hlb_handle h, double out[4]);

/* hlb_monitor without any device allocation.  It has no counterpart in the
 * reference: it is for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc).  The per-workgroup partials and the four results live in a
 * fixed array of the library's own device memory, hlb_noalloc_scratch_bytes()
 * = 16 MiB per GPU, held until the process ends; a lattice of more than
 * 2,097,120 active slabs needs more partials than it holds and gets
 * HLB_ERANGE (hlb_monitor serves it).  Results equal hlb_monitor's bit for
 * bit.  Every handle on a GPU shares the array: calls that overlap on one
 * GPU race. */
int hlb_monitor_noalloc(hlb_handle h, double out[4]);
int64_t hlb_noalloc_scratch_bytes(void);

/* Iolet state (outlet = 0: inlet `index`, 1: outlet `index`):
 * out[0] density used by the last step's ghost sites (for Windkessel iolets,
 * the committed density), out[1] densityNew, out[2] flowRate, out[3]
 * flowRateOld -- the members of InOutLetWK3 (src/lb/iolets/InOutLetWK3.h)
 * read by BoundaryValues::GetBoundaryDensity (BoundaryValues.cc:211-214). */
int hlb_iolet_state(hlb_handle h, int outlet, int index, double out[4]);

/* ---- lattice tables (LatticeData accessors, for parity and extraction) -- */
int64_t hlb_site_count(hlb_handle h);          /* GetLocalFluidSiteCount */
/* Get{MidDomain,DomainEdge}CollisionCount (LatticeData.h:375-436). */
int hlb_class_counts(hlb_handle h, int64_t out[6]);
/* GetGlobalSiteCoords (LatticeData.h:611-614), n*3. */
int hlb_site_coords(hlb_handle h, int64_t* out);
/* The reference's push table GetStreamedIndex (LatticeData.h:516-520,
 * LatticeData.cc:366-443): n*19 int64, rubbish slot n*19, rebuilt from the
 * device pull table.  pull may be NULL; else it receives the device pull
 * table (18 rows of n uint32: source site of direction j = 1..18, or the
 * site itself where a boundary condition supplies the value). */
int hlb_neighbour_tables(hlb_handle h, int64_t* push, uint32_t* pull);
/* SiteData masks, ioletId and SiteType (src/geometry/SiteDataBare.cc:24-76). */
int hlb_site_masks(hlb_handle h, uint32_t* wall, uint32_t* iolet, int32_t* iolet_id,
                   int32_t* site_type);
/* GetCutDistance (n*18, double) and GetNormalToWall (n*3, double). */
int hlb_wall_geometry(hlb_handle h, double* dist, double* normal);

/* ---- iolet tables from files ------------------------------------------ */
/* InOutLetFile::CalculateTable (src/lb/iolets/InOutLetFile.cc:37-101) and
 * InOutLetFileVelocity::CalculateTable (InOutLetFileVelocity.cc:31-90): reads
 * "time value" pairs (s; mmHg or m/s), clips them to total_steps *
 * time_step with an interpolated end point, and fills out[0..total_steps]
 * with the lattice density (pressure) or lattice speed (velocity) of each
 * step, the profile repeating as the reference repeats it.  out_len must be
 * at least total_steps + 1.  For pressure, *density_min receives
 * GetDensityMin (may be NULL). */
int hlb_iolet_file_table(const char* path, int velocity, int64_t total_steps, double time_step, double voxel_size,
                         double* out, int64_t out_len, double* density_min);

/* ---- procedural geometries (the inputs a .gmy file would hold) ---------- */
typedef struct hlb_geom hlb_geom;
typedef struct hlb_iolet_geom {
  int32_t is_inlet;
  int32_t id;
  double position[3];
  double normal[3]; /* points into the fluid */
  double radius;
} hlb_iolet_geom;

/* Straight voxelised cylinder along z: radius r, length L sites, axis at the
 * centre of a box_xy x box_xy cross-section; inlet at z = -0.5, outlet at
 * z = L - 0.5. */
int hlb_geom_cylinder(double radius, int32_t length, int32_t box_xy, hlb_geom** out);
/* Symmetric Y-bifurcation: parent (radius rp, length lp) along +z, two
 * daughters (radius rd, length ld) at +-angle_deg in the x-z plane; radii
 * carry a seeded smooth jitter of relative amplitude jitter. */
int hlb_geom_ybifurcation(double rp, double lp, double rd, double ld, double angle_deg,
                          double jitter, uint64_t seed, hlb_geom** out);
/* Straight pipe with a Gaussian stenosis of the given area reduction at
 * mid-length, width parameter w (lattice units). */
int hlb_geom_stenosed_pipe(double radius, int32_t length, double area_reduction, double width,
                           hlb_geom** out);
/* Binary tree of tapering tubes in a box (multiples of 8): the root (radius
 * root_radius) enters at the z = -0.5 face along +z, every segment end splits
 * into two children of radius taper * r turned by U(angle_min, angle_max)
 * degrees to opposite sides of a random plane, segments are length_factor *
 * r long (shortened to stay two radii inside the box).  generations levels
 * give 2^generations - 1 segments; inlet 0 at the root, outlets 0.. at the
 * leaves.  Voxelised on nthreads host threads (0: all cores); the result
 * does not depend on the thread count. */
int hlb_geom_vessel_tree(uint64_t seed, int32_t generations, double root_radius, double taper,
                         double length_factor, double angle_min_deg, double angle_max_deg,
                         const int32_t box[3], int32_t nthreads, hlb_geom** out);
/* Reads a HemeLB geometry file, version 4 (gmy_plus = 1: the .gmy+ variant
 * with per-block weights); replaces GeometryReader::LoadAndDecompose's
 * reading (src/geometry/GeometryReader.cc:382-446, 851-935) on one process.
 * The file carries no iolet positions (they come from the XML): the returned
 * geometry lists none. */
int hlb_geom_read_gmy(const char* path, int gmy_plus, hlb_geom** out);
/* Fills the view with pointers into g (valid until hlb_geom_free). */
int hlb_geom_view(const hlb_geom* g, hlb_geometry* view);
int hlb_geom_iolets(const hlb_geom* g, hlb_iolet_geom* out, int max_iolets);
void hlb_geom_free(hlb_geom* g);

#ifdef __cplusplus
}
#endif

#endif /* HEMEPURE_AMD_H */
