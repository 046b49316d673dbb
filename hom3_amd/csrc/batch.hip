// Batched solves: many independent first-order Euler instances of uneven
// size (each with its own grid, 2:1 refinement and time step) advanced by
// one persistent kernel per RK stage, with the whole step captured in a
// hipGraph and the launch shape picked by a timing autotuner.
//
// There is no batching in the reference; each instance follows the single
// solver's step exactly (solver.hpp:140-145: set_dt, evolve, advance) with
// its own dt, time and step, so a batch of one equals hom3g_solver_solve.
//
// Layout.  Every instance's internal cells start at a multiple of the tile
// size, each instance keeping its own (Morton leaf) order: one SoA state
// array per stage buffer, and one list of tiles (tile.hpp) whose headers name
// their instance.  Zero-gradient Neumann and periodic ghosts are read through
// the cells they copy, so no ghost-fill pass is needed.
//
// A fixed grid of workgroups sweeps the tiles (persistent kernel); the final
// stage also reduces each tile's CFL bound of the new state into its
// instance's running minimum (atomic min on an order-preserving integer
// encoding, exact and order independent) and advances time and step.
#include <algorithm>
#include <cstring>

#include "tile.hpp"

namespace hom3g {

namespace {

inline unsigned nblk(int64_t n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

// compute_dt (solver.hpp:511-517) of the current FP64 state, per instance
template <int ND>
__global__ void __launch_bounds__(kTileCells) k_batch_dt(TileView t, const double* U, long long ld, DevScalars* scal,
                                                         PhysConst pc) {
  constexpr int NV = ND + 2;
  __shared__ double red[kTileCells / 64];
  for (long long tile = blockIdx.x; tile < t.ntile; tile += gridDim.x) {
    const TileHdr H = t.hdr[tile];
    const long long c = tile * kTileCells + threadIdx.x;
    double m = 1.7976931348623157e308;
    if ((int)threadIdx.x < H.n) {
      double q[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) q[v] = U[v * ld + c];
      m = ref_min(m, cell_dt_fast<ND, false>(q, __builtin_ldexp(H.root, -(int)t.lev[c]), pc));
    }
    for (int o = 32; o > 0; o >>= 1) m = ref_min(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int k = 1; k < kTileCells / 64; ++k) m = ref_min(m, red[k]);
      lower_dt(scal[H.inst], m);
    }
    __syncthreads();
  }
}

// per instance: set_dt (solver.hpp:541-551) and reset of the running minimum
__global__ void k_batch_set_dt(int n, DevScalars* s) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  DevScalars& S = s[i];
  const double dtm = dt_minimum(S);
  if (S.time + S.dt < S.tEnd) S.dt = (S.step == S.forced_step) ? S.forced_dt : dtm;
  else S.dt = S.tEnd - S.time;
  reset_dt(S);
}

__global__ void k_batch_reset(int n, DevScalars* s) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) reset_dt(s[i]);
}

// forward Euler's lhs = rhs copy (solver.hpp:473-476)
__global__ void k_batch_copy(const double* __restrict__ a, double* __restrict__ b, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    b[i] = a[i];
}

void launch_stage(Ctx& C, BatchDev& B, int kind, const void* in, bool in32, void* out, bool out32, bool last,
                  StepDt dt_mode = StepDt::set) {
  tile_stage(C, B.nd, tile_view(B.tiles), B.pc,
             TileStage{in, B.U.p, out, in32, out32, (long long)B.ld, (long long)B.ld, kind, last, last, dt_mode},
             B.scal.p,
             (unsigned)std::min<long long>(B.grid, B.tiles.ntile));
}

void launch_dt(Ctx& C, BatchDev& B) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min<long long>(B.grid, B.tiles.ntile)), dim3(kTileCells), 0, C.stream,
                       tile_view(B.tiles), (const double*)B.U.p, (long long)B.ld, B.scal.p, B.pc);
    H3_LAUNCH_CHECK();
  };
  if (B.nd == 2) go(k_batch_dt<2>);
  else go(k_batch_dt<3>);
}

void drop_graph(BatchDev& B) {
  if (B.exec) (void)hipGraphExecDestroy(B.exec);
  if (B.graph) (void)hipGraphDestroy(B.graph);
  B.exec = nullptr;
  B.graph = nullptr;
}

// One step of every instance (solver.hpp:140-145): [compute_dt] set_dt,
// evolve (solver.hpp:469-499 + SSP-RK3), advance.  After the first step the
// CFL bound of the new state comes fused out of the last stage, which also
// advances.
void enqueue_step(Ctx& C, BatchDev& B) {
  // SSP-RK3 stages on few tiles set the dt themselves (StepDt)
  const bool own_dt = B.ti == HOM3G_TI_SSP_RK3 && B.tiles.ntile <= kOwnDtTiles;
  if (!own_dt) {
    hipLaunchKernelGGL(k_batch_set_dt, dim3(nblk(B.ninst)), dim3(256), 0, C.stream, B.ninst, B.scal.p);
    H3_LAUNCH_CHECK();
  }
  const bool f32 = B.precision == HOM3G_FP32_STATE;
  void* s1 = f32 ? (void*)B.S1f.p : (void*)B.S1d.p;
  void* s2 = f32 ? (void*)B.S2f.p : (void*)B.S2d.p;
  if (B.ti == HOM3G_TI_SSP_RK3) {
    launch_stage(C, B, 0, B.U.p, false, s1, f32, false, own_dt ? StepDt::first : StepDt::set);
    launch_stage(C, B, 2, s1, f32, s2, f32, false, own_dt ? StepDt::middle : StepDt::set);
    launch_stage(C, B, 3, s2, f32, B.U.p, false, true, own_dt ? StepDt::last : StepDt::set);
  } else if (B.ti == HOM3G_TI_HEUN_RK2) {
    launch_stage(C, B, 0, B.U.p, false, s1, f32, false);
    launch_stage(C, B, 1, s1, f32, B.U.p, false, true);
  } else {
    launch_stage(C, B, 0, B.U.p, false, B.S1d.p, false, true);
    const long long n = (long long)B.nvars * B.ld;
    hipLaunchKernelGGL(k_batch_copy, dim3(2048), dim3(256), 0, C.stream, (const double*)B.S1d.p, B.U.p, n);
    H3_LAUNCH_CHECK();
  }
}

void build_graph(Ctx& C, BatchDev& B) {
  if (B.exec) return;
  hipGraph_t g = nullptr;
  H3_HIP(hipStreamBeginCapture(C.stream, hipStreamCaptureModeThreadLocal));
  try {
    enqueue_step(C, B);
  } catch (...) {
    (void)hipStreamEndCapture(C.stream, &g);
    if (g) (void)hipGraphDestroy(g);
    throw;
  }
  H3_HIP(hipStreamEndCapture(C.stream, &g));
  B.graph = g;
  H3_HIP(hipGraphInstantiate(&B.exec, B.graph, nullptr, nullptr, 0));
}

void ensure_dtmin(Ctx& C, BatchDev& B) {
  if (B.dtmin_current) return;
  hipLaunchKernelGGL(k_batch_reset, dim3(nblk(B.ninst)), dim3(256), 0, C.stream, B.ninst, B.scal.p);
  H3_LAUNCH_CHECK();
  launch_dt(C, B);
  B.dtmin_current = true;
}

}  // namespace

void batch_create(Ctx& C, const std::vector<SolverDev*>& inst, int precision, BatchDev& B) {
  H3_REQUIRE(!inst.empty(), "empty batch");
  const SolverDev& S0 = *inst[0];
  B.nd = S0.nd;
  B.nvars = S0.nvars;
  B.ninst = (int)inst.size();
  B.precision = precision;
  B.ti = S0.P.ti;
  B.pc = S0.pc;
  for (SolverDev* S : inst) {
    H3_REQUIRE(S->built, "batch instance not built");
    H3_REQUIRE(S->P.physics == HOM3G_EULER && S->P.flux == HOM3G_FLUX_AUSM && S->P.recon == HOM3G_RECON_NONE,
               "batched instances must be first-order Euler AUSM");
    H3_REQUIRE(S->nd == B.nd && S->P.ti == B.ti && S->P.gamma == S0.P.gamma && S->P.cfl == S0.P.cfl,
               "batched instances must share nd, time integration, gamma and CFL");
    for (const BCDesc& b : S->bcs) {
      H3_REQUIRE(b.kind == HOM3G_BC_PERIODIC || zero_gradient(b), "batched instances support zero-gradient Neumann and periodic boundaries only");
    }
  }
  B.off.resize(B.ninst);
  B.nint.resize(B.ninst);
  std::vector<TileHdr> hdr;
  std::vector<long long> tile0(B.ninst + 1);
  int64_t N = 0;
  for (int i = 0; i < B.ninst; ++i) {
    tile0[i] = (long long)hdr.size();
    B.off[i] = tile0[i] * kTileCells;
    B.nint[i] = inst[i]->n_int;
    N += inst[i]->n_int;
    H3_REQUIRE(tile_count(C, *inst[i], hdr, i), "batched instance has a face without neighbour");
  }
  tile0[B.ninst] = (long long)hdr.size();
  H3_REQUIRE(tile0[B.ninst] * kTileCells < INT32_MAX / 2, "too many cells in the batch for 32-bit ids");
  H3_REQUIRE(tile_place(C, B.nd, hdr, B.tiles), "too many tile faces in the batch for 32-bit offsets");
  B.ncell = N;
  B.ld = B.tiles.ntile * kTileCells;
  const int nv = B.nvars;
  const size_t total = (size_t)nv * B.ld;
  B.U.alloc(total);
  H3_HIP(hipMemsetAsync(B.U.p, 0, total * sizeof(double), C.stream));  // the cells past an instance's end
  if (precision == HOM3G_FP32_STATE) {
    B.S1f.alloc(total);
    B.S2f.alloc(total);
    H3_HIP(hipMemsetAsync(B.S1f.p, 0, total * sizeof(float), C.stream));
    H3_HIP(hipMemsetAsync(B.S2f.p, 0, total * sizeof(float), C.stream));
    if (B.ti == HOM3G_TI_EULER_FWD) B.S1d.alloc(total);
  } else {
    B.S1d.alloc(total);
    B.S2d.alloc(total);
    H3_HIP(hipMemsetAsync(B.S2d.p, 0, total * sizeof(double), C.stream));
  }
  if (B.S1d.p) H3_HIP(hipMemsetAsync(B.S1d.p, 0, total * sizeof(double), C.stream));
  B.scal.alloc(B.ninst);
  for (int i = 0; i < B.ninst; ++i) {
    SolverDev& S = *inst[i];
    H3_HIP(hipMemcpy2DAsync(B.U.p + B.off[i], (size_t)B.ld * sizeof(double), S.lhs.p, (size_t)S.cap * sizeof(double),
                            (size_t)S.n_int * sizeof(double), nv, hipMemcpyDeviceToDevice, C.stream));
    H3_HIP(hipMemcpyAsync(B.scal.p + i, S.scal.p, sizeof(DevScalars), hipMemcpyDeviceToDevice, C.stream));
    tile_fill(C, S, B.tiles, tile0[i], tile0[i + 1] - tile0[i]);
  }
  H3_HIP(hipStreamSynchronize(C.stream));
  // default launch shape until autotuned
  int dev = 0, ncu = 0;
  H3_HIP(hipGetDevice(&dev));
  H3_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  B.ncu = ncu > 0 ? ncu : 256;
  B.grid = B.ncu * 64;
  B.dtmin_current = false;
}

void batch_set_config(Ctx& C, BatchDev& B, int block, int tile, int grid) {
  H3_REQUIRE(block >= 64 && block <= 512 && block % 64 == 0, "block must be a multiple of 64 in [64, 512]");
  H3_REQUIRE(tile >= block, "tile must hold at least one cell per thread");
  H3_REQUIRE(grid >= 1, "grid must be positive");
  (void)C;
  B.grid = grid;
  drop_graph(B);
}

void batch_solve(Ctx& C, BatchDev& B, int nsteps, bool use_graph) {
  H3_REQUIRE(nsteps >= 0, "nsteps must be non-negative");
  if (nsteps == 0) return;
  ensure_dtmin(C, B);
  if (!use_graph) {
    for (int s = 0; s < nsteps; ++s) enqueue_step(C, B);
    return;
  }
  build_graph(C, B);
  for (int s = 0; s < nsteps; ++s) H3_HIP(hipGraphLaunch(B.exec, C.stream));
}

// Times candidate numbers of workgroups on stage 1 of the current state with
// the current dt (written to a stage buffer: neither the state nor the
// instances' scalars change) and keeps the fastest.
void batch_autotune(Ctx& C, BatchDev& B, int* best_block, int* best_tile, int* best_grid, float* best_ms) {
  const bool f32 = B.precision == HOM3G_FP32_STATE;
  void* s1 = f32 ? (void*)B.S1f.p : (void*)B.S1d.p;
  // up to 64 workgroups per CU: about one tile per workgroup, the persistent
  // sweep degenerating to a plain launch
  const int wgs_per_cu[] = {2, 3, 4, 6, 8, 16, 64};
  float bms = 1e30f;
  int bg = B.grid;
  for (int w : wgs_per_cu) {
    batch_set_config(C, B, kTileCells, kTileCells, B.ncu * w);
    launch_stage(C, B, 0, B.U.p, false, s1, f32, false);  // warm
    float tmin = 1e30f;
    for (int r = 0; r < 5; ++r) {
      H3_HIP(hipEventRecord(C.ev0, C.stream));
      launch_stage(C, B, 0, B.U.p, false, s1, f32, false);
      H3_HIP(hipEventRecord(C.ev1, C.stream));
      H3_HIP(hipEventSynchronize(C.ev1));
      float ms = 0;
      H3_HIP(hipEventElapsedTime(&ms, C.ev0, C.ev1));
      tmin = std::min(tmin, ms);
    }
    if (tmin < bms) { bms = tmin; bg = B.grid; }
  }
  batch_set_config(C, B, kTileCells, kTileCells, bg);
  if (best_block) *best_block = kTileCells;
  if (best_tile) *best_tile = kTileCells;
  if (best_grid) *best_grid = bg;
  if (best_ms) *best_ms = bms;
}

// events around nsteps steps (graph or stream launches), ms per step
float batch_time_solve(Ctx& C, BatchDev& B, int nsteps, bool use_graph) {
  ensure_dtmin(C, B);
  if (use_graph) build_graph(C, B);  // capture outside the timed region
  H3_HIP(hipEventRecord(C.ev0, C.stream));
  batch_solve(C, B, nsteps, use_graph);
  H3_HIP(hipEventRecord(C.ev1, C.stream));
  H3_HIP(hipEventSynchronize(C.ev1));
  float ms = 0;
  H3_HIP(hipEventElapsedTime(&ms, C.ev0, C.ev1));
  return nsteps > 0 ? ms / nsteps : 0.f;
}

void batch_download(Ctx& C, BatchDev& B, int inst, double* out) {
  H3_REQUIRE(inst >= 0 && inst < B.ninst, "instance out of range");
  const int64_t n = B.nint[inst];
  for (int v = 0; v < B.nvars; ++v)
    H3_HIP(hipMemcpyAsync(out + (size_t)v * n, B.U.p + (size_t)v * B.ld + B.off[inst], n * sizeof(double),
                          hipMemcpyDeviceToHost, C.stream));
  H3_HIP(hipStreamSynchronize(C.stream));
}

void batch_scalars(Ctx& C, BatchDev& B, int inst, DevScalars* out) {
  H3_REQUIRE(inst >= 0 && inst < B.ninst, "instance out of range");
  H3_HIP(hipMemcpyAsync(out, B.scal.p + inst, sizeof(DevScalars), hipMemcpyDeviceToHost, C.stream));
  H3_HIP(hipStreamSynchronize(C.stream));
}

void batch_release(BatchDev& B) { drop_graph(B); }

}  // namespace hom3g
