// Host-side data structures of the hom3g library (device buffers, grids,
// solvers, the context).  Not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <memory>
#include <string>
#include <vector>

#include "../../include/hom3g.h"
#include "memory.hpp"
#include "physics.hpp"

namespace hom3g {

// Scalars of one solver kept in device memory so the step loop never
// synchronises with the host (solver.hpp:406-416).
//
// The running CFL minimum is spread over kDtSlots places in lines of their
// own: the workgroups that are resident first all lower it, and atomics on
// one address serialise (about 12 ns each).  With one place they took 3.4 of
// the 32 us of a 256^2 vortex step, 3% of a 2048^2 one and 1.5% of the
// channel's.
constexpr int kDtSlots = 8;
struct alignas(128) DtSlot {
  unsigned long long v;  // ordered-int encoded (dbl_to_ordered)
};
struct DevScalars {
  double dt, time, tEnd, forced_dt;
  long long step, forced_step;
  double dtdx;               // dt / h on a uniform grid (brick steps), set with dt
  long long diverged_step;   // first step whose dt left [1e-300, 1e300] (utilities.hpp:73-76), -1: none
  double pub_dt, pub_dtdx;   // the dt of the step under way, from its first stage to its last (StepDt)
  DtSlot dtmin[kDtSlots];
};
__host__ __device__ __forceinline__ double dt_minimum(const DevScalars& s) {
  unsigned long long m = s.dtmin[0].v;
#pragma unroll
  for (int k = 1; k < kDtSlots; ++k) m = s.dtmin[k].v < m ? s.dtmin[k].v : m;
  return ordered_to_dbl(m);
}
__device__ __forceinline__ void reset_dt(DevScalars& s) {
#pragma unroll
  for (int k = 0; k < kDtSlots; ++k) s.dtmin[k].v = dbl_to_ordered(1.7976931348623157e308);
}
// By one thread of a workgroup.  Eight workgroups in a row, one on each XCD,
// share a place, so that every place sees all parts of the grid and falls as
// soon as one of them reaches the minimum.  A place per XCD (workgroup mod 8)
// is lowered by that XCD's share of the bricks alone: where the bound falls
// along it every workgroup comes with an atomic (a step of the 2048^2 vortex
// in FP32 states 233-244 us, so 210; with a single place 226; 48 batch
// instances 568 -> 527 us; 32^3 Taylor-Green 31.0 -> 31.1).
__device__ __forceinline__ void lower_dt(DevScalars& s, double m) {
  atomic_lower(&s.dtmin[blockIdx.x / 8 % kDtSlots].v, m);
}

// Where a stage kernel gets its step's dt.  SSP-RK3 on bricks and tiles needs
// no kernel for set_dt (solver.hpp:541-551): every workgroup of the first
// stage forms the dt from the scalars (which that launch does not change) and
// one publishes it in pub_dt, the second stage resets the running minimum
// (which the first read and the third lowers), and the last makes it dt and
// advances.  A launch of its own cost 1.8 us and a gap of about 2 on small
// grids (of 36 us a step on the 256^2 vortex), 4.7 us after large stages.
// (256^2 vortex 35.9 -> 32.3 us a step.)  With many workgroups the launch is
// the cheaper one: 16,384 bricks (2048^2 vortex, FP32 states) took 4% longer
// without it and 4,096 (128^3) 1%, 256 gained 10%; 19,409 tiles (5 M-leaf
// blast) took 3% longer, 6,912 gained 5% and 3,191 nothing.
constexpr long long kOwnDtBricks = 2048, kOwnDtTiles = 8192;
enum class StepDt : int { set = 0, first = 1, middle = 2, last = 3 };  // set: k_set_dt or a coupling kernel has set it

// what the step's dt is formed from: loaded ahead of its use (vector loads: a
// wait for scalar ones would be taken with the next LDS read's)
struct DtInputs {
  double time, dt, tEnd, forced_dt;
  long long step, forced_step;
  unsigned long long m[kDtSlots];
};
template <class T>
__device__ __forceinline__ T load_own(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
__device__ __forceinline__ DtInputs load_dt_inputs(const DevScalars* s) {
  DtInputs i;
  i.time = load_own(&s->time);
  i.dt = load_own(&s->dt);
  i.tEnd = load_own(&s->tEnd);
  i.forced_dt = load_own(&s->forced_dt);
  i.step = load_own(&s->step);
  i.forced_step = load_own(&s->forced_step);
#pragma unroll
  for (int k = 0; k < kDtSlots; ++k) i.m[k] = load_own(&s->dtmin[k].v);
  return i;
}
__device__ __forceinline__ double step_dt(const DtInputs& i) {
  unsigned long long m = i.m[0];
#pragma unroll
  for (int k = 1; k < kDtSlots; ++k) m = i.m[k] < m ? i.m[k] : m;
  if (i.time + i.dt < i.tEnd) return (i.step == i.forced_step) ? i.forced_dt : ordered_to_dbl(m);
  return i.tEnd - i.time;
}
// (h: the cell length of a brick solver, 0 otherwise)
__device__ __forceinline__ void publish_dt(DevScalars* s, double dt, double h) {
  // solution_diverged (utilities.hpp:73-76), checked by the solve driver; the
  // end-time clamp (run_solver stops there) is not divergence
  if (s->time + s->dt < s->tEnd && (dt < 1e-300 || dt > 1e300) && s->diverged_step < 0) s->diverged_step = s->step;
  s->pub_dt = dt;
  s->pub_dtdx = h > 0.0 ? dt / h : 0.0;
}
// one thread of the stage's launch (per instance); dt: the step's
__device__ __forceinline__ void step_scalars(DevScalars* s, StepDt m, bool advance, double dt, double h) {
  if (m == StepDt::first) publish_dt(s, dt, h);
  if (m == StepDt::middle) reset_dt(*s);
  if (m == StepDt::last) {
    s->dt = dt;
    s->dtdx = s->pub_dtdx;
  }
  // advance (solver.hpp:502-505): no stage but the first reads time or step
  if (advance) {
    s->time += dt;
    s->step += 1;
  }
}

struct GridDev {
  int nd = 0;
  int max_solvers = 1;
  double root_len = 0, root_x[3] = {0, 0, 0};
  int64_t nnodes = 0;
  int uniform_level = -1;  // >=0 when generated by MinLevel from the root
  DevBuf<int64_t> parent, first_child;
  DevBuf<int32_t> level;
};

struct BCDesc {
  int kind = 0;
  hom3g_geometry geom{};
  double params[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int nparams = 0;
  int other_sid = -1;
  double kratio = 1.0;
  // HOM3G_BC_HOST_CALLBACK: the condition, its user data and its slope hook
  hom3g_bc_callback cb = nullptr;
  void* user = nullptr;
  int hook = HOM3G_SLOPE_DEFAULT;
};

// The ghosts a host-callback condition fills (apply-range order), their
// boundary cells and centres, cached at their first fill
struct HostBCRun {
  int bc = -1;
  std::vector<int64_t> ghosts, bndry;   // cell ids
  std::vector<double> xg, xb;           // nd x m, column-major
  DevBuf<int32_t> dg, db;
};

constexpr int kMaxBC = 16;

// BC descriptor table passed by value to kernels
struct BCTable {
  int nbc;
  int kind[kMaxBC];
  double params[kMaxBC][8];
  int nparams[kMaxBC];
  double kratio[kMaxBC];
  const double* other_lhs[kMaxBC];
  long long other_ld[kMaxBC];
  double other_gamma[kMaxBC];
  int other_physics[kMaxBC];
};

// One captured solver step (hipGraph); solver_solve replays it while the
// key (buffers, kernel, physics, boundary conditions) is unchanged
struct StepGraph {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  uint64_t key = 0;
  StepGraph() = default;
  StepGraph(const StepGraph&) = delete;
  StepGraph& operator=(const StepGraph&) = delete;
  StepGraph(StepGraph&& o) noexcept : graph(o.graph), exec(o.exec), key(o.key) {
    o.graph = nullptr;
    o.exec = nullptr;
    o.key = 0;
  }
  void drop() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    exec = nullptr;
    graph = nullptr;
    key = 0;
  }
  ~StepGraph() { drop(); }
};

// zero-gradient Neumann: the ghost holds a copy of its boundary cell
inline bool zero_gradient(const BCDesc& b) {
  if (b.kind != HOM3G_BC_NEUMANN) return false;
  for (int k = 0; k < b.nparams; ++k)
    if (b.params[k] != 0.0) return false;
  return true;
}

// Tiles (tile.hpp): runs of kTileCells consecutive cells with their face lists
constexpr int kTileCells = 256;
struct TileHdr {
  int32_t halo0, ext0;  // the tile's first entries in halo_more and ext_more
  int32_t inst;         // whose scalars (batches)
  int32_t pad;
  uint16_t n, nh;       // cells, halo cells
  uint16_t ne[3];       // extra faces per direction
  uint16_t first;       // first tile of its instance
  double root, inv_root;  // cell length of level 0 and its reciprocal
};
struct TileTab {
  DevBuf<TileHdr> hdr;
  DevBuf<uint32_t> face, ext, ext_more;
  DevBuf<uint8_t> lev;
  DevBuf<int32_t> halo, halo_more;
  long long ntile = 0;
  void release() {
    hdr.release();
    for (DevBuf<uint32_t>* b : {&face, &ext, &ext_more}) b->release();
    lev.release();
    for (DevBuf<int32_t>* b : {&halo, &halo_more}) b->release();
    ntile = 0;
  }
};

struct SolverDev {
  int id = -1, grid_id = -1, solver_idx = 0;
  hom3g_physics P{};
  PhysConst pc{};
  int nd = 0, nvars = 0, npos = 0;
  int64_t ncells = 0, n_int = 0, n_ghost = 0, cap = 0;
  bool built = false;
  // domain
  hom3g_geometry domain_geom{};
  int domain_sign = 0;
  std::vector<uint8_t> domain_mask;
  std::vector<BCDesc> bcs;
  // state (SoA, ld = cap)
  DevBuf<double> lhs, rhs, stg, lhs_old;
  DevBuf<double> slopes;  // table-driven CNS: each cell's slopes of the stage input (nd x nv x cap)
  DevBuf<float> rhs32, stg32;
  // topology
  DevBuf<int32_t> nghbr;        // npos x cap, -1 = none, <= -2: face towards finer cells
  DevBuf<int32_t> fine;         // 2^(nd-1) finer cells per fine face (f = -(v + 2))
  int64_t nfine = 0;
  bool nonuniform = false;      // leaves of more than one level
  uint64_t perturb_seed = 0;    // seeded density perturbation after the IC
  double perturb_amp = 0;
  DevBuf<int64_t> node_idx;     // cap
  DevBuf<int32_t> bc_idx;       // cap
  DevBuf<double> x_center;      // nd x cap
  DevBuf<double> length;        // cap
  DevBuf<double> dist;          // npos x cap
  DevBuf<int64_t> node2cell;    // nnodes of the grid
  // per ghost (index g - n_int)
  DevBuf<int32_t> g_bndry, g_pos, g_hookbc, g_applybc, g_image, g_partner;
  DevBuf<double> g_dist;
  DevBuf<double> source;
  DevBuf<DevScalars> scal;
  DevScalars host_scal{};
  // brick kernel eligibility
  bool brick_ok = false;
  bool brick_table = false;     // tiled bricks: halos from brick_halo (brick_table_build)
  DevBuf<uint32_t> brick_halo;  // per brick, the cells of its halo list
  DevBuf<int32_t> brick_rev_rp, brick_rev_src;  // per cell, the halo entries that read it (CSR)
  DevBuf<int32_t> brick_rev_tl;                 // the cells read by some halo entry
  int64_t brick_rev_nt = 0;
  int level = -1;               // uniform level
  int face_mode[3][2] = {{0, 0}, {0, 0}, {0, 0}};  // 0 clamp (zero-gradient), 1 periodic
  bool uses_vortex_bc = false;
  bool partners_built = false;
  bool dtmin_current = false;   // scal.dtmin holds the CFL minimum of the current lhs
  double h_uniform = 0;         // cell length of a uniform grid
  int kernel = HOM3G_KERNEL_GENERIC;
  bool tile_ok = false;         // first-order Euler stages on tiles (tile.hpp)
  bool tile_ghosts = false;     // some tile reads ghosts: filled before every stage
  TileTab tile;
  StepGraph step_graph;
  // host-callback boundary conditions (staging of the ghosts they fill)
  bool has_host_bc = false, host_bc_ready = false;
  std::vector<std::unique_ptr<HostBCRun>> host_bc_runs;
  DevBuf<double> hbc_dev;
  PinnedBuf<double> hbc_pin;
  PinnedBuf<DevScalars> hbc_scal;
};

// Batched instances (batch.hip): each instance's internal cells from a
// multiple of the tile size on, one list of tiles over all of them
struct BatchDev {
  int nd = 0, nvars = 0, ninst = 0, precision = HOM3G_FP64, ti = HOM3G_TI_SSP_RK3;
  PhysConst pc{};
  int64_t ncell = 0, ld = 0;    // cells of all instances; leading dimension of the state
  DevBuf<double> U, S1d, S2d;   // nv x ld, FP64 state and stage buffers
  DevBuf<float> S1f, S2f;       // FP32 stage buffers
  TileTab tiles;
  DevBuf<DevScalars> scal;      // per instance
  std::vector<int64_t> off, nint;
  int ncu = 256, grid = 1024;
  bool dtmin_current = false;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

struct Ctx {
  Pool pool;                // kept between adjoint calls
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::vector<std::unique_ptr<GridDev>> grids;
  std::vector<std::unique_ptr<SolverDev>> solvers;
  std::vector<std::unique_ptr<BatchDev>> batches;
  DevBuf<double> red;            // reduction scratch
  DevBuf<unsigned long long> red_u64;
  int ckpt_memory = 0;           // HOM3G_CKPT_*: where the adjoint keeps its checkpoints
  double* scratch = nullptr;     // this device's address of the static scratch (noalloc_init)
  // optional per-stage-launch event timing (hom3g_solver_profile_solve)
  bool prof_on = false;
  std::vector<hipEvent_t> prof_events;
  size_t prof_used = 0;
  void prof_mark() {
    if (!prof_on) return;
    if (prof_used == prof_events.size()) {
      hipEvent_t e;
      H3_HIP(hipEventCreate(&e));
      prof_events.push_back(e);
    }
    H3_HIP(hipEventRecord(prof_events[prof_used++], stream));
  }
};

// topology.hip
void grid_generate_uniform(Ctx& C, GridDev& G, int level);
void grid_compute_levels(Ctx& C, GridDev& G);
void grid_neighbors(Ctx& C, GridDev& G, int64_t* host_out);
void grid_geometry(Ctx& C, GridDev& G, double* x_rowmajor, double* len);
int64_t grid_refine_region(Ctx& C, GridDev& G, int max_level, const hom3g_geometry& g, double band);
int64_t grid_balance(Ctx& C, GridDev& G);
void solver_build(Ctx& C, GridDev& G, SolverDev& S);
void solver_build_partners(Ctx& C, SolverDev& S);

// tile.hip: the solver's tiles when its stages can run on them
void solver_build_tiles(Ctx& C, SolverDev& S);

// stepper.hip
void solver_alloc_state(Ctx& C, SolverDev& S);
void solver_impose_ic(Ctx& C, SolverDev& S, int kind, const double* params, int np);
void solver_init_time(Ctx& C, SolverDev& S);
void solver_solve(Ctx& C, SolverDev& S, int nsteps);
// one step (solver.hpp:140-145)
struct StepFlags {
  bool skip_dt_reduction = false;  // the dt is forced for this step
  bool dt_set = false;             // set_dt is done (couple_cht_step, force_pair_dt)
  bool lhs_ghosts = false;         // the ghosts of lhs are those of its current state
  // the caller may read the lhs ghosts after this step (they hold apply_bcs of
  // the state the step began with: tiles that read no ghost leave them to the
  // last step of a solve)
  bool last = true;
};
void solver_step(Ctx& C, SolverDev& S, const StepFlags& f);
// a prescribed dt for the coupled pair's next step, set (StepFlags::dt_set);
// rec: device memory for the two dts taken, or null
void force_pair_dt(Ctx& C, SolverDev& cns, SolverDev& heat, double dt, double scaling, double* rec);
void solver_min_dt_device(Ctx& C, SolverDev& S, unsigned long long* out_dev);
double solver_min_dt(Ctx& C, SolverDev& S);
void solver_conservation_sums(Ctx& C, SolverDev& S, double* out);
// set-up of the static device scratch on the context's device, and the sums
// that use it instead of allocating (sums_dev: device memory, stream-ordered)
void noalloc_init(Ctx& C);
void solver_conservation_sums_noalloc(Ctx& C, SolverDev& S, double* sums_dev);
int64_t solver_check_state(Ctx& C, SolverDev& S);
void solver_pull_scalars(Ctx& C, SolverDev& S);
void solver_push_scalars(Ctx& C, SolverDev& S);
void couple_cht_step(Ctx& C, SolverDev& cns, SolverDev& heat, double Tr0);
void couple_same_step(Ctx& C, SolverDev& a, SolverDev& b);
BCTable make_bc_table(Ctx& C, SolverDev& S, int role = 0);
void solver_fill_ghosts(Ctx& C, SolverDev& S, double* buf);
void solver_fill_ghosts(Ctx& C, SolverDev& S, float* buf);
// impose_initial_condition (solver.hpp:980-992) with a host callback
// evaluated at every internal cell's Gauss points
void solver_impose_ic_host(Ctx& C, SolverDev& S, hom3g_ic_callback f, void* user);
float copy_calibration(Ctx& C, int64_t bytes);
float copy_bandwidth(Ctx& C, int64_t bytes, int variant, int grid, int block, int reps);
void solver_apply_perturbation(Ctx& C, SolverDev& S);

// adjoint.hip
struct ChtRunStats {
  double J = 0;
  float ms_forward = 0, ms_reverse = 0, ms_primal_step = 0;
};
// obs (host, one value per internal solid cell) selects the final-state
// misfit J = 1/2 sum (T_N - obs)^2 instead of the wall heat flux
void cht_objective_run(Ctx& C, SolverDev& cns, SolverDev& heat, double Tr0, int nsteps, const double* dts,
                       double* dts_out, ChtRunStats& st, const double* obs = nullptr);
void cht_tangent_run(Ctx& C, SolverDev& cns, SolverDev& heat, double Tr0, int nsteps, const double* dts,
                     const double* dsource, double* J, double* dJ, const double* obs = nullptr);
void cht_adjoint_run(Ctx& C, SolverDev& cns, SolverDev& heat, double Tr0, int nsteps, const double* dts,
                     int ckpt_every, double* grad_source, ChtRunStats& st, const double* obs = nullptr);

// batch.hip
void batch_create(Ctx& C, const std::vector<SolverDev*>& inst, int precision, BatchDev& B);
void batch_set_config(Ctx& C, BatchDev& B, int block, int tile, int grid);
void batch_solve(Ctx& C, BatchDev& B, int nsteps, bool use_graph);
void batch_autotune(Ctx& C, BatchDev& B, int* block, int* tile, int* grid, float* ms);
float batch_time_solve(Ctx& C, BatchDev& B, int nsteps, bool use_graph);
void batch_download(Ctx& C, BatchDev& B, int inst, double* out);
void batch_scalars(Ctx& C, BatchDev& B, int inst, DevScalars* out);
void batch_release(BatchDev& B);

// brick.hip
bool brick_supported(const SolverDev& S);
bool brick_table_build(Ctx& C, SolverDev& S);
void brick_stage(Ctx& C, SolverDev& S, int stage, const void* in, void* out, bool fuse_dt, bool advance,
                 StepDt dt_mode);

}  // namespace hom3g
