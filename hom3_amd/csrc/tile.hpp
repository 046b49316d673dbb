// Tiles: runs of kTileCells consecutive cells of a solver's leaf order with
// their faces listed, for the first-order Euler stages on any grid
// (tile.hip builds the lists and runs the stages; batch.hip concatenates the
// lists of its instances).
#pragma once
#include "internal.hpp"

namespace hom3g {

// Halo cells held in LDS (NHC) and extra faces per direction and chunk (CE).
// 3D FP64: 51 KB of LDS, three workgroups per CU.  On the 5 M-leaf refined
// blast a tile has 336 halo cells and 47-72 extra faces per direction in the
// median (95%: 368 and 80).  With 320 and 64 the blast took 25% longer (0.8 M
// leaves) and 14% longer (5 M): too many tiles then read halo cells from
// memory and take two chunks; with 384 and 256 or 512 and 128 it took 11-18%
// longer at 0.8 M (fewer workgroups per CU).  A 2D tile of 16 x 16 cells has
// 64 and 16, but the coarse side of a level interface up to 490 and 225, and
// a small batch waits for those tiles: 12 instances took 5.0 ms with 128 and
// 64, 4.4 with 256 and 128, 3.7 with 256 and 256 (FP64, 41 KB, three
// workgroups per CU); 48 instances 25.5-25.8 ms (FP32 states) with each.
template <int ND> struct TileCfg;
template <> struct TileCfg<3> { static constexpr int NHC = 384, CE = 128; };
template <> struct TileCfg<2> { static constexpr int NHC = 256, CE = 256; };

// The lists of all tiles as the kernels read them.  The first NHC halo cells
// and CE extra faces of a tile are at places of their own, so that their
// loads need not wait for the header; the rest follow the offsets in it.
struct TileView {
  const TileHdr* hdr;
  const uint32_t* face;   // nd x ldw: lower-face position | upper-face slot << 16
  const uint8_t* lev;     // ldw: level of every cell
  const int32_t* halo;    // ntile x NHC, padded with the tile's first cell
  const uint32_t* ext;    // ntile x nd x CE
  const int32_t* halo_more;
  const uint32_t* ext_more;
  long long ntile, ldw;
};

inline TileView tile_view(const TileTab& t) {
  return TileView{t.hdr.p, t.face.p, t.lev.p, t.halo.p, t.ext.p, t.halo_more.p, t.ext_more.p,
                  t.ntile, t.ntile * (long long)kTileCells};
}

// Workgroups of a stage: one per tile up to 64 per CU, a sweep past that (5 M
// leaves: 19,409 tiles 22.7 ms a pass with one each, 21.7 with 16,384 or
// 8,192, 23.7 with 2,048: the dispatch of workgroups costs more than the
// uneven last turn)
inline unsigned tile_grid(long long ntile) { return (unsigned)(ntile < 64 * 256 ? ntile : 64 * 256); }

// Appends the headers of S's tiles (lists not yet placed) with their list lengths; false if some cell has a side without
// neighbour or ghost.
bool tile_count(Ctx& C, const SolverDev& S, std::vector<TileHdr>& hdr, int inst);
// Places the lists of all headers (halo0, ext0) and allocates the table;
// false if they exceed 32-bit offsets.
bool tile_place(Ctx& C, int nd, std::vector<TileHdr>& hdr, TileTab& t);
// Fills the lists of S's tiles, headers [tile0, tile0 + n); S's cells are
// the cells tile0 * kTileCells onwards of the state arrays.
void tile_fill(Ctx& C, const SolverDev& S, TileTab& t, long long tile0, long long n);

// One RK stage over all tiles (kind: see TileArgs); in/out are double or,
// for FP32 stage states, float.
struct TileStage {
  const void* in;
  const double* base;
  void* out;
  bool in32, out32;
  long long ld, ncell;  // leading dimension; cells of the arrays that may be read
  int kind;
  bool fuse_dt;   // reduce the CFL bound of the new state into each instance's running minimum
  bool advance;   // last stage of the step: also time += dt, ++step of each instance
  StepDt dt_mode;
};
void tile_stage(Ctx& C, int nd, const TileView& t, const PhysConst& pc, const TileStage& a, DevScalars* scal,
                unsigned grid);

}  // namespace hom3g
