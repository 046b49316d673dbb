// First-order Euler stages (AUSM) on tiles of consecutive cells, for refined
// grids, ragged domains and batches: every grid the bricks do not cover.
//
// The leaf order keeps siblings together and runs along the Morton curve
// inside a level, so kTileCells consecutive cells are a few compact blocks.
// One workgroup takes one tile: the tile's cells and the cells behind its
// outer faces (the halo list) go to LDS with their primitives, every face is
// evaluated once, and the cells sum their faces' fluxes.  The table-driven
// kernel gathers six neighbours per cell, forms seven sets of primitives and
// evaluates every face from both sides; here a cell costs 1.8-2 sets of
// primitives and 3.4-3.6 faces (3D), and a face towards finer cells occupies
// only its own lanes instead of every lane of its wave.
//
// Faces.  Per direction, the face below cell i (towards one cell: local,
// halo or the coarser neighbour) is evaluated by thread i into slot i.  The
// faces that no cell of the tile has below itself are "extra": the upper
// faces of the tile's outer cells, an upper face towards a coarser cell, and
// the 2^(nd-1) sub-faces of a face towards finer cells.  They are listed per
// direction in cell order and evaluated by one wave (another one in each
// direction), in chunks of CE.
//
// Measured (one MI355X, refined blast, per step of three stages): 0.82 M
// leaves FP64 0.24 -> 0.148 ms, 4.97 M leaves FP32 states 0.67 -> 0.455 ms
// against the table-driven kernel and its separate ghost fills, CFL
// reduction and advance; per cell-stage 490-600 VALU instead of 1,000 (FP64).
// A tile takes 7-9 us, 60% of it waiting: the chain from the halo list to the
// halo states to the first face, and the two barriers per direction; at 5 M
// leaves the stages read and write 5.2-5.5 TB/s (the halo cells are read 1.3
// times per cell on top of the compulsory bytes, in part from the caches), a
// device copy 4.9.  FP64 holds three workgroups per CU (LDS and 168
// VGPRs; at 174 it held two and the 0.82 M-leaf step took 0.18 ms), FP32 four
// (118-123 VGPRs; held to 96 or 80 it spills and runs 13% and 60% slower).
//
// 2D batches (which evaluated every face from both sides too), per step:
// 512 instances of 76.7 M cells FP64 7.05 -> 6.25 ms, FP32 states 5.59 ->
// 4.32 ms; a pass of 40 steps of 12 instances (base grids 64^2 to 256^2, FP64)
// 4.47 -> 3.42 ms.
//
// Boundaries.  A zero-gradient Neumann ghost holds a copy of its boundary
// cell and a periodic one a copy of its image, so their faces read that cell
// and need no ghost; other ghosts are halo cells, filled before the stage.
#include <algorithm>
#include <type_traits>

#include "tile.hpp"

namespace hom3g {

namespace {

constexpr int T = kTileCells;
constexpr unsigned kFineFlag = 0x8000u;

// ---- building the lists ------------------------------------------------------

struct TileTopo {
  const int32_t* nghbr;
  const int32_t* fine;
  const int32_t* g_apply;
  const int32_t* g_image;
  const double* len;
  double root;
  long long ld, n_int;
  int kind[kMaxBC];  // 1: zero-gradient Neumann, 2: periodic, 0: other
};

struct TileOut {
  TileHdr* hdr;
  uint32_t* face;
  uint8_t* lev;
  int32_t *halo, *halo_more;
  uint32_t *ext, *ext_more;
  long long ldw, cell0;
};

constexpr int kMissing = INT32_MIN;

// what cell c meets across side pos: a cell (>= 0; itself for a zero-gradient
// ghost, the image for a periodic one, otherwise the ghost), a face towards
// finer cells (<= -2) or nothing (kMissing)
__device__ __forceinline__ int across(const TileTopo& t, long long c, int pos) {
  const int raw = t.nghbr[pos * t.ld + c];
  if (raw == -1) return kMissing;
  if (raw < t.n_int) return raw;
  const int g = raw - (int)t.n_int;
  const int b = t.g_apply[g];
  const int k = b >= 0 ? t.kind[b] : 0;
  return k == 1 ? (int)c : (k == 2 ? t.g_image[g] : raw);
}

__device__ __forceinline__ int block_scan(int v, int* sh, int& total) {
  const int i = threadIdx.x;
  sh[i] = v;
  __syncthreads();
  for (int o = 1; o < T; o <<= 1) {
    const int w = i >= o ? sh[i - o] : 0;
    __syncthreads();
    sh[i] += w;
    __syncthreads();
  }
  total = sh[T - 1];
  const int r = sh[i] - v;
  __syncthreads();
  return r;
}

// FILL false: the list lengths of every tile (hdr.nh, hdr.ne); true: the lists
template <int ND, bool FILL>
__global__ void __launch_bounds__(T) k_tile_lists(TileTopo t, TileOut o, long long tile0, int* missing) {
  __shared__ int sh[T];
  constexpr int K = 1 << (ND - 1);
  const long long tile = tile0 + blockIdx.x;
  const int i = threadIdx.x;
  const long long base = (long long)blockIdx.x * T;
  const int n = (int)(t.n_int - base < T ? t.n_int - base : T);
  const bool has = i < n;
  const long long c = base + i;
  int nh = 0;
  constexpr int NHC = TileCfg<ND>::NHC, CE = TileCfg<ND>::CE;
  const TileHdr H = FILL ? o.hdr[tile] : TileHdr{};
  int more0 = H.ext0;
  auto put_halo = [&](int h, int cell) {
    if (h < NHC) o.halo[tile * NHC + h] = (int32_t)(cell + o.cell0);
    else o.halo_more[H.halo0 + h - NHC] = (int32_t)(cell + o.cell0);
  };
  // (len = root / 2^level, exact; lanes past the last cell: level 0, and below
  // their own slots for both faces)
  if (FILL) o.lev[tile * T + i] = has ? (uint8_t)ilogb(t.root / t.len[c]) : (uint8_t)0;
  for (int d = 0; d < ND; ++d) {
    const int lo = has ? across(t, c, 2 * d) : (int)c, up = has ? across(t, c, 2 * d + 1) : (int)c;
    if (has && (lo == kMissing || up == kMissing)) atomicOr(missing, 1);
    auto local = [&](int x) { return x >= base && x < base + n; };
    const bool lo_fine = has && lo <= -2 && lo != kMissing, up_fine = has && up <= -2 && up != kMissing;
    // the face above c is the face below its upper neighbour if that one is
    // in the tile and meets c below
    const bool shared = has && up >= 0 && local(up) && up != (int)c && across(t, up, 2 * d) == (int)c;
    const int n_lo = lo_fine ? K : 0, n_up = !has || shared ? 0 : (up_fine ? K : 1);
    const int groups = (lo_fine ? 1 : 0) + (up_fine ? 1 : 0), single = n_up == 1 ? 1 : 0;
    // halo cells: the lower neighbour, then those of the extra faces, each
    // group in cell order
    const bool lo_halo = has && lo >= 0 && !local(lo);
    int tot;
    const int h_lo = block_scan(lo_halo ? 1 : 0, sh, tot);
    const int halo_lo = nh;
    nh += tot;
    int nhx = 0;
    auto sub = [&](int side, int k) {  // other cell of extra face k of a side
      const int v = side ? up : lo;
      return v >= 0 ? v : t.fine[(long long)(-(v + 2)) * K + k];
    };
    for (int k = 0; k < n_lo; ++k) nhx += local(sub(0, k)) ? 0 : 1;
    for (int k = 0; k < n_up; ++k) nhx += local(sub(1, k)) ? 0 : 1;
    const int h_x = block_scan(nhx, sh, tot);
    const int halo_x = nh;
    nh += tot;
    // extra faces: the groups of K sub-faces first, so that no group is split
    // between chunks, then the single ones
    int g0 = block_scan(groups, sh, tot);
    const int ng = tot;
    const int s0 = K * ng + block_scan(single, sh, tot);
    const int ne = K * ng + tot;
    if constexpr (FILL) {
      if (has) {
        unsigned lower = 0, upper;
        if (lo_fine) {}
        else if (local(lo)) lower = (unsigned)(lo - base);
        else {
          lower = (unsigned)(T + halo_lo + h_lo);
          put_halo(halo_lo + h_lo, lo);
        }
        int h = halo_x + h_x;
        int start[2] = {K * g0, 0};
        if (lo_fine) ++g0;
        start[1] = up_fine ? K * g0 : s0;
        for (int side = 0; side < 2; ++side) {
          const int m = side ? n_up : n_lo;
          for (int k = 0; k < m; ++k) {
            const int x = sub(side, k);
            unsigned pos;
            if (local(x)) pos = (unsigned)(x - base);
            else {
              put_halo(h, x);
              pos = (unsigned)(T + h++);
            }
            const int e = start[side] + k;
            uint32_t* to = e < CE ? &o.ext[(tile * ND + d) * CE + e] : &o.ext_more[more0 + e - CE];
            *to = (unsigned)i | ((unsigned)side << 8) | (pos << 16);
          }
        }
        if (lo_fine) lower = kFineFlag | (unsigned)start[0];
        if (shared) upper = (unsigned)(up - base);
        else upper = up_fine ? (kFineFlag | (unsigned)start[1]) : (unsigned)(T + start[1]);
        o.face[d * o.ldw + tile * T + i] = lower | (upper << 16);
      } else {
        o.face[d * o.ldw + tile * T + i] = (unsigned)i | ((unsigned)i << 16);
      }
    } else if (i == 0) {
      o.hdr[tile].ne[d] = (uint16_t)ne;
    }
    more0 += ne > CE ? ne - CE : 0;
  }
  if (FILL)
    for (int h = nh + i; h < NHC; h += T) put_halo(h, (int)base);
  if (!FILL && i == 0) {
    o.hdr[tile].nh = (uint16_t)nh;
    o.hdr[tile].n = (uint16_t)n;
  }
}

TileTopo tile_topo(Ctx& C, const SolverDev& S) {
  TileTopo t;
  t.nghbr = S.nghbr.p;
  t.fine = S.fine.p;
  t.g_apply = S.g_applybc.p;
  t.g_image = S.g_image.p;
  t.len = S.length.p;
  t.root = C.grids[S.grid_id]->root_len;
  t.ld = S.cap;
  t.n_int = S.n_int;
  for (int b = 0; b < kMaxBC; ++b) {
    t.kind[b] = 0;
    if (b >= (int)S.bcs.size()) continue;
    const BCDesc& d = S.bcs[b];
    if (d.kind == HOM3G_BC_PERIODIC) t.kind[b] = 2;
    else if (zero_gradient(d)) t.kind[b] = 1;
  }
  return t;
}

// ---- stages ------------------------------------------------------------------

struct TileArgs {
  TileView t;
  const void* in;
  const double* base;
  void* out;
  long long ld, ncell;
  int kind;  // 0: in+nf  1: 0.5*((base+in)+nf)  2: 0.75 base + 0.25 (in+nf)  3: 1/3 base + 2/3 (in+nf)  4: in+nf
  int fuse_dt, advance, stream;
  StepDt dt_mode;
  DevScalars* scal;
};

template <int ND, class TC>
struct TileSmem {
  static constexpr int NV = ND + 2, NP = T + TileCfg<ND>::NHC;
  TC q[NV][NP];
  TC p[NP], iar[NP];                    // p and 1 / (rho a)
  TC f[NV][T + TileCfg<ND>::CE];        // face fluxes of one direction
  double red[T / 64];
};

template <int ND, class TC>
struct CellState {
  TC q[ND + 2], p, iar;
};

template <int ND, class TC, class TIn>
__device__ __forceinline__ void load_state(const TileArgs& A, long long c, TC* q) {
#pragma unroll
  for (int v = 0; v < ND + 2; ++v) q[v] = TC(static_cast<const TIn*>(A.in)[v * A.ld + c]);
}

// U^n is read once per stage and the output is not read again by it: past
// the caches when the state does not fit them (TileArgs::stream)
__device__ __forceinline__ double load_base(const TileArgs& A, long long k) {
  return A.stream ? __builtin_nontemporal_load(&A.base[k]) : A.base[k];
}
template <class TOut>
__device__ __forceinline__ void store_out(const TileArgs& A, long long k, TOut x) {
  TOut* p = static_cast<TOut*>(A.out) + k;
  if (A.stream) __builtin_nontemporal_store(x, p);
  else *p = x;
}

// Workgroups go round-robin to the 8 XCDs, each with its own L2: runs of 8
// consecutive tiles to one XCD, so that half of a tile's halo is in its L2
// (3% on the 0.8 M-leaf blast, 1.5% at 5 M against the plain order; one
// eighth of the tiles per XCD was slower at 5 M leaves).  A bijection on
// [0, n).
__device__ __forceinline__ long long xcd_run(long long b, long long n) {
  constexpr long long R = 8, P = 8 * R;
  if (b >= n / P * P) return b;
  const long long r = b % P;
  return b - r + (r % 8) * R + r / 8;
}

template <int ND, class TC, class TIn>
__device__ __forceinline__ void fetch(const TileSmem<ND, TC>& s, const TileArgs& A, const PhysConst& pc, int halo0,
                                      int pos, CellState<ND, TC>& w) {
  if (__builtin_expect(pos >= T + TileCfg<ND>::NHC, 0)) {
    load_state<ND, TC, TIn>(A, A.t.halo_more[halo0 + pos - T - TileCfg<ND>::NHC], w.q);
    euler_prims<ND, TC>(w.q, TC(pc.gamma), TC(pc.gm1), w.p, w.iar);
    return;
  }
#pragma unroll
  for (int v = 0; v < ND + 2; ++v) w.q[v] = s.q[v][pos];
  w.p = s.p[pos];
  w.iar = s.iar[pos];
}

template <int ND, int D, class TC>
__device__ __forceinline__ void tile_flux(const CellState<ND, TC>& L, const CellState<ND, TC>& R, TC gamma, TC* f) {
  ausm_flux_fast<ND, D, TC>(L.q, L.q[D], L.p, gamma * L.p * L.iar, L.iar, R.q, R.q[D], R.p, gamma * R.p * R.iar,
                            R.iar, f);
}

// the extra face of a chunk this thread evaluates in direction D
template <int D>
__device__ __forceinline__ int ext_lane() {
  return ((int)threadIdx.x - 64 * (D + 1)) & (T - 1);
}

// one direction: the fluxes of its faces into the slots, then every cell's sum
template <int ND, int D, class TC, class TIn>
__device__ __forceinline__ void tile_direction(TileSmem<ND, TC>& s, const TileArgs& A, const PhysConst& pc,
                                               const TileHdr& H, int more0, unsigned face, unsigned ext, bool has,
                                               const CellState<ND, TC>& own, TC* acc) {
  constexpr int NV = ND + 2, CE = TileCfg<ND>::CE, K = 1 << (ND - 1);
  const int i = threadIdx.x;
  const TC gamma = TC(pc.gamma);
  const unsigned lower = face & 0xffffu, upper = face >> 16;
  const int ne = H.ne[D];
  if (has && !(lower & kFineFlag)) {
    CellState<ND, TC> L;
    fetch<ND, TC, TIn>(s, A, pc, H.halo0, (int)lower, L);
    TC f[NV];
    tile_flux<ND, D, TC>(L, own, gamma, f);
#pragma unroll
    for (int v = 0; v < NV; ++v) s.f[v][i] = f[v];
  }
  // the fluxes below and above the cell, each complete before they are
  // subtracted: they nearly cancel
  TC fm[NV], fp[NV];
  for (int e0 = 0;; e0 += CE) {
    // extra faces [e0, e0 + CE) by consecutive lanes from wave D + 1 on
    const int k = ext_lane<D>();
    if (k < CE && e0 + k < ne) {
      const unsigned x = e0 == 0 ? ext : A.t.ext_more[more0 + e0 - CE + k];
      CellState<ND, TC> a, b;
      fetch<ND, TC, TIn>(s, A, pc, H.halo0, (int)(x & 0xffu), a);
      fetch<ND, TC, TIn>(s, A, pc, H.halo0, (int)(x >> 16), b);
      const bool up = (x >> 8) & 1u;  // the other cell is above
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const TC lo = up ? a.q[v] : b.q[v], hi = up ? b.q[v] : a.q[v];
        a.q[v] = lo;
        b.q[v] = hi;
      }
      const TC pl = up ? a.p : b.p, ph = up ? b.p : a.p, il = up ? a.iar : b.iar, ih = up ? b.iar : a.iar;
      a.p = pl; b.p = ph; a.iar = il; b.iar = ih;
      TC f[NV];
      tile_flux<ND, D, TC>(a, b, gamma, f);
#pragma unroll
      for (int v = 0; v < NV; ++v) s.f[v][T + k] = f[v];
    }
    __syncthreads();
    // the mean of the sub-faces of a face towards finer cells, summed in
    // pairs (equal sub-fluxes give exactly their value)
    auto finer = [&](unsigned group, TC* g) {
      const int x = T + (int)(group & ~kFineFlag) - e0;
      if (x < T || x >= T + CE) return;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        TC sum = s.f[v][x] + s.f[v][x + 1];
        if constexpr (K == 4) sum += s.f[v][x + 2] + s.f[v][x + 3];
        g[v] = sum * TC(1.0 / K);
      }
    };
    const bool lo_fine = (lower & kFineFlag) != 0, up_fine = (upper & kFineFlag) != 0;
    if (e0 == 0) {
      const bool here = upper < (unsigned)(T + CE);  // a slot of the tile or of this chunk
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        fm[v] = lo_fine ? TC(0) : s.f[v][i];
        fp[v] = here ? s.f[v][here ? upper : 0] : TC(0);
      }
    } else if (upper >= (unsigned)(T + e0) && upper < (unsigned)(T + e0 + CE)) {
#pragma unroll
      for (int v = 0; v < NV; ++v) fp[v] = s.f[v][upper - e0];
    }
    if (lo_fine) finer(lower, fm);
    if (up_fine) finer(upper, fp);
    __syncthreads();
    if (e0 + CE >= ne) {
#pragma unroll
      for (int v = 0; v < NV; ++v) acc[v] += fm[v] - fp[v];
      break;
    }
  }
}

template <int ND, class TC, class TIn, class TOut>
__global__ void __launch_bounds__(T, ND == 3 && sizeof(TC) == 8 ? 3 : 4) k_tile_stage(TileArgs A, PhysConst pc) {
  constexpr int NV = ND + 2, NHC = TileCfg<ND>::NHC, CE = TileCfg<ND>::CE;
  __shared__ TileSmem<ND, TC> s;
  const int i = threadIdx.x;
  for (long long b = blockIdx.x; b < A.t.ntile; b += gridDim.x) {
    const long long tile = xcd_run(b, A.t.ntile);
    // everything whose place follows from the tile's number is in flight
    // before the header is needed: the tile's cells, their faces, the halo
    // list and this thread's extra face of each direction (a load inside a
    // pass would hold up the whole workgroup)
    const long long c = tile * T + i;
    const long long cl = c < A.ncell ? c : A.ncell - 1;
    CellState<ND, TC> own;
    load_state<ND, TC, TIn>(A, cl, own.q);
    int hid[(NHC + T - 1) / T];
#pragma unroll
    for (int r = 0; r * T < NHC; ++r) hid[r] = A.t.halo[tile * NHC + (r * T + i < NHC ? r * T + i : 0)];
    unsigned face[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) face[d] = A.t.face[d * A.t.ldw + c];
    const int lev = A.t.lev[c];
    unsigned ext[3] = {0, 0, 0};
    const uint32_t* ex = A.t.ext + tile * ND * CE;
    if (ext_lane<0>() < CE) ext[0] = ex[ext_lane<0>()];
    if (ext_lane<1>() < CE) ext[1] = ex[CE + ext_lane<1>()];
    if (ND == 3 && ext_lane<2>() < CE) ext[2] = ex[2 * CE + ext_lane<2>()];
    const TileHdr H = A.t.hdr[tile];
    const bool has = i < H.n;
    DevScalars* S = A.scal + H.inst;
    double dt = A.dt_mode == StepDt::set ? S->dt : S->pub_dt;
#pragma unroll
    for (int r = 0; r * T < NHC; ++r) {
      const int j = r * T + i;
      if (j < NHC && j < H.nh) {
        CellState<ND, TC> w;
        load_state<ND, TC, TIn>(A, hid[r], w.q);
        euler_prims<ND, TC>(w.q, TC(pc.gamma), TC(pc.gm1), w.p, w.iar);
#pragma unroll
        for (int v = 0; v < NV; ++v) s.q[v][T + j] = w.q[v];
        s.p[T + j] = w.p;
        s.iar[T + j] = w.iar;
      }
    }
    euler_prims<ND, TC>(own.q, TC(pc.gamma), TC(pc.gm1), own.p, own.iar);
#pragma unroll
    for (int v = 0; v < NV; ++v) s.q[v][i] = own.q[v];
    s.p[i] = own.p;
    s.iar[i] = own.iar;
    __syncthreads();
    // U^n, in flight during the passes
    double bq[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) bq[v] = (A.kind >= 1 && A.kind <= 3) ? load_base(A, v * A.ld + cl) : 0.0;
    TC acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = TC(0);
    auto more = [&](int d) { return H.ne[d] > CE ? H.ne[d] - CE : 0; };
    int more0 = H.ext0;
    tile_direction<ND, 0, TC, TIn>(s, A, pc, H, more0, face[0], ext[0], has, own, acc);
    more0 += more(0);
    if constexpr (ND == 3) {
      tile_direction<ND, 1, TC, TIn>(s, A, pc, H, more0, face[1], ext[1], has, own, acc);
      more0 += more(1);
    }
    double qd[NV];  // FP64 input of an FP32 stage, read again (cached)
    if constexpr (sizeof(TIn) != sizeof(TC)) {
#pragma unroll
      for (int v = 0; v < NV; ++v) qd[v] = static_cast<const double*>(A.in)[v * A.ld + cl];
    }
    tile_direction<ND, ND - 1, TC, TIn>(s, A, pc, H, more0, face[ND - 1], ext[ND - 1], has, own, acc);

    if (A.dt_mode == StepDt::first) dt = step_dt(load_dt_inputs(S));
    const double dtdx = dt * __builtin_ldexp(H.inv_root, lev);
    // The RK combinations with their fused products fixed.  In U/3 + 2/3 s
    // it matters which product is rounded: (1/3) U rounded and 2/3 s fused
    // leaves 60 steps of the 0.8 M-leaf blast 6.0e-16 from the FP64
    // reference, the other way round 1.4e-15 (against long double on 51 k
    // leaves 3.3e-16 and 9.2e-16; the table-driven kernel 3.4e-16).
    double o[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      // the stage input at its stored type: an FP64 one does not lose the
      // digits that the FP32 flux arithmetic does without
      const double q = sizeof(TIn) == sizeof(TC) ? (double)own.q[v] : qd[v];
      const double sv = __builtin_fma(dtdx, (double)acc[v], q);
      switch (A.kind) {
        case 1: o[v] = 0.5 * (bq[v] + sv); break;
        case 2: o[v] = __builtin_fma(0.75, bq[v], 0.25 * sv); break;
        case 3: o[v] = __builtin_fma(2. / 3., sv, (1. / 3.) * bq[v]); break;
        default: o[v] = sv; break;
      }
      if (has) store_out<TOut>(A, v * A.ld + c, TOut(o[v]));
    }
    if (A.fuse_dt) {
      double m = 1.7976931348623157e308;
      if (has) {
        double qo[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) qo[v] = (double)TOut(o[v]);
        m = ref_min(m, cell_dt_fast<ND, false>(qo, __builtin_ldexp(H.root, -lev), pc));
      }
      for (int k = 32; k > 0; k >>= 1) m = ref_min(m, __shfl_xor(m, k, 64));
      if ((i & 63) == 0) s.red[i >> 6] = m;
      __syncthreads();
      if (i == 0) {
        for (int k = 1; k < T / 64; ++k) m = ref_min(m, s.red[k]);
        lower_dt(*S, m);
      }
    }
    // the scalars, by one tile per instance
    if (H.first && i == 0) step_scalars(S, A.dt_mode, A.advance != 0, dt, 0.0);
    // (no barrier here: the next tile writes the states only past this
    // tile's last closing barrier, and the reduction's values only past its
    // own barriers)
  }
}

}  // namespace

bool tile_count(Ctx& C, const SolverDev& S, std::vector<TileHdr>& hdr, int inst) {
  const long long n = (S.n_int + T - 1) / T;
  DevBuf<TileHdr> h;
  DevBuf<int> missing;
  h.alloc(n);
  missing.alloc(1);
  int zero = 0;
  missing.upload(&zero, 1, C.stream);
  TileOut o{h.p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
  if (S.nd == 2)
    hipLaunchKernelGGL((k_tile_lists<2, false>), dim3((unsigned)n), dim3(T), 0, C.stream, tile_topo(C, S), o, 0ll,
                       missing.p);
  else
    hipLaunchKernelGGL((k_tile_lists<3, false>), dim3((unsigned)n), dim3(T), 0, C.stream, tile_topo(C, S), o, 0ll,
                       missing.p);
  H3_LAUNCH_CHECK();
  std::vector<TileHdr> v(n);
  h.download(v.data(), n, C.stream);
  missing.download(&zero, 1, C.stream);
  H3_HIP(hipStreamSynchronize(C.stream));
  if (zero) return false;
  const double root = C.grids[S.grid_id]->root_len;
  for (long long k = 0; k < n; ++k) {
    TileHdr& H = v[k];
    H.inst = inst;
    H.first = k == 0 ? 1 : 0;
    if (S.nd == 2) H.ne[2] = 0;
    H.root = root;
    H.inv_root = 1.0 / root;
    hdr.push_back(H);
  }
  return true;
}

bool tile_place(Ctx& C, int nd, std::vector<TileHdr>& hdr, TileTab& t) {
  const int NHC = nd == 2 ? TileCfg<2>::NHC : TileCfg<3>::NHC, CE = nd == 2 ? TileCfg<2>::CE : TileCfg<3>::CE;
  long long nh = 0, ne = 0;
  for (TileHdr& H : hdr) {
    H.halo0 = (int32_t)nh;
    H.ext0 = (int32_t)ne;
    nh += std::max(0, (int)H.nh - NHC);
    for (int d = 0; d < nd; ++d) ne += std::max(0, (int)H.ne[d] - CE);
  }
  if (nh >= INT32_MAX || ne >= INT32_MAX) return false;
  t.ntile = (long long)hdr.size();
  t.hdr.alloc(hdr.size());
  t.hdr.upload(hdr.data(), hdr.size(), C.stream);
  t.face.alloc((size_t)nd * t.ntile * T);
  t.lev.alloc((size_t)t.ntile * T);
  t.halo.alloc((size_t)t.ntile * NHC);
  t.ext.alloc((size_t)t.ntile * nd * CE);
  t.halo_more.alloc(std::max<long long>(1, nh));
  t.ext_more.alloc(std::max<long long>(1, ne));
  H3_HIP(hipStreamSynchronize(C.stream));
  return true;
}

void tile_fill(Ctx& C, const SolverDev& S, TileTab& t, long long tile0, long long n) {
  TileOut o{t.hdr.p, t.face.p, t.lev.p, t.halo.p, t.halo_more.p, t.ext.p, t.ext_more.p, t.ntile * (long long)T,
            tile0 * T};
  if (S.nd == 2)
    hipLaunchKernelGGL((k_tile_lists<2, true>), dim3((unsigned)n), dim3(T), 0, C.stream, tile_topo(C, S), o, tile0,
                       (int*)nullptr);
  else
    hipLaunchKernelGGL((k_tile_lists<3, true>), dim3((unsigned)n), dim3(T), 0, C.stream, tile_topo(C, S), o, tile0,
                       (int*)nullptr);
  H3_LAUNCH_CHECK();
}

// First-order Euler AUSM off the bricks, unless the table-driven kernel is
// asked for.  Not with the
// isentropic-vortex condition (its fill rewrites boundary cells, so a CFL
// bound fused into the last stage would be stale), host callbacks or
// Euler-Euler coupling (their ghosts come from outside the solver), nor
// where a cell has a side without neighbour or ghost (the table-driven
// kernel poisons such a cell).
void solver_build_tiles(Ctx& C, SolverDev& S) {
  S.tile_ok = false;
  if (S.kernel != HOM3G_KERNEL_GENERIC || S.P.kernel == HOM3G_KERNEL_GENERIC || S.P.physics != HOM3G_EULER ||
      S.P.flux != HOM3G_FLUX_AUSM || S.P.recon != HOM3G_RECON_NONE || S.has_host_bc || S.uses_vortex_bc)
    return;
  S.tile_ghosts = false;
  for (const BCDesc& b : S.bcs) {
    if (b.kind == HOM3G_BC_EULER_COUPLING) return;
    if (b.kind != HOM3G_BC_PERIODIC && !zero_gradient(b)) S.tile_ghosts = true;
  }
  std::vector<TileHdr> hdr;
  try {
    if (!tile_count(C, S, hdr, 0) || !tile_place(C, S.nd, hdr, S.tile)) return;
  } catch (const OutOfMemory&) {
    // the lists are 21 (2D) or 25 B (3D) per cell on top of the solver's tables and states,
    // which are in place: it steps without them
    S.tile.release();
    return;
  }
  tile_fill(C, S, S.tile, 0, S.tile.ntile);
  S.tile_ok = true;
}

void tile_stage(Ctx& C, int nd, const TileView& t, const PhysConst& pc, const TileStage& a, DevScalars* scal,
                unsigned grid) {
  // past the caches once the arrays of a stage exceed half of the 256 MB MALL:
  // 4% faster on 5 M leaves (FP32 states, 400 MB a stage), 3% slower on 0.8 M
  // (FP64, 100 MB), whose arrays stay there from stage to stage
  const double bytes = (double)a.ncell * (nd + 2) * ((a.in32 ? 4 : 8) + (a.out32 ? 4 : 8) + (a.kind ? 8 : 0));
  TileArgs A{t, a.in, a.base, a.out, a.ld, a.ncell, a.kind, a.fuse_dt ? 1 : 0, a.advance ? 1 : 0,
             bytes > 128.0 * (1 << 20) ? 1 : 0, a.dt_mode, scal};
  auto go = [&](auto kern) {
    C.prof_mark();
    hipLaunchKernelGGL(kern, dim3(grid), dim3(T), 0, C.stream, A, pc);
    H3_LAUNCH_CHECK();
    C.prof_mark();
  };
  auto by_type = [&](auto ndc) {
    constexpr int ND = decltype(ndc)::value;
    if (!a.in32 && !a.out32) go(k_tile_stage<ND, double, double, double>);
    else if (!a.in32) go(k_tile_stage<ND, float, double, float>);
    else if (a.out32) go(k_tile_stage<ND, float, float, float>);
    else go(k_tile_stage<ND, float, float, double>);
  };
  if (nd == 2) by_type(std::integral_constant<int, 2>());
  else by_type(std::integral_constant<int, 3>());
}

}  // namespace hom3g
