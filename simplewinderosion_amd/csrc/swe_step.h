// swe_step.h -- argument blocks of the tile-owned step kernel (swe_step.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace swe {

// Tile shapes of the step kernel: SX x SY cells (x the slow axis), NT
// threads, a register budget that keeps WPE waves per SIMD.  Every shape
// computes the same bits; swe_autotune times them (SWE_TUNE_SHAPE).
struct StepShape {
  int32_t sx, sy, threads, waves;
};
constexpr int kStepShapes = 5;
constexpr StepShape kStepShape[kStepShapes] = {
    {16, 32, 256, 5},  // default: the best measured on the 1024^2 and 64-terrain workloads
    {32, 16, 256, 5},
    {16, 16, 128, 5},
    {16, 32, 256, 4},
    {32, 32, 512, 4},
};
constexpr int kStepChunk = 32;                 // tiles per chunk sum of the input counts

// Halo of the cells that the colour-ordered relax of a tile and its one-cell
// halo can depend on: a cascade reads and writes its 3 x 3 block, so a
// dependence runs through cells of decreasing class at most two cells apart.
// Away from the extra classes of a periodic axis, with classes x-major, x
// changes only between the three x classes and y in every step, which gives
// (-4 .. +6) x (-10 .. +18) around a cell.  A region that meets one of the
// last n mod 3 cells of a periodic axis sees up to five classes an axis:
// (-5 .. +6) x (-14 .. +24) when no axis has two such cells and both are at
// least 16 cells, (-6 .. +6) x (-26 .. +30) otherwise.  The extents, one
// larger each way for the tile's one-cell halo, are checked against the full
// dependence sets in tests/test_colour_halo.py.
struct ColourHalo {
  int32_t xl, xh, yl, yh;
};
constexpr ColourHalo kColourHalo = {5, 7, 11, 19};
constexpr ColourHalo kColourHaloSeam = {6, 7, 15, 25};
constexpr ColourHalo kColourHaloMax = {7, 7, 27, 31};
inline ColourHalo colour_halo(int32_t nx, int32_t ny, bool periodic) {
  if (!periodic || (nx % 3 == 0 && ny % 3 == 0)) return kColourHalo;
  return nx % 3 <= 1 && ny % 3 <= 1 && nx >= 16 && ny >= 16 ? kColourHaloSeam : kColourHaloMax;
}

// Dynamic LDS of k_colour_step: the region's masters, events, list and
// classes, or the march's accumulators
inline int64_t colour_lds(const StepShape& sh, const ColourHalo& h, bool track, int32_t layers) {
  const int64_t ry = sh.sy + h.yl + h.yh, r = (sh.sx + h.xl + h.xh) * ry;
  const int64_t relax = r * (8 * layers + 4 + 2 + 1) + 2 * (ry + 8);
  const int64_t march = (int64_t)sh.sx * sh.sy * (8 * layers + 4 + (track ? 32 : 0));
  return ((relax > march ? relax : march) + 15) / 16 * 16;
}

// Workgroups of k_colour_step that the chip's 256 CUs hold at once: four waves
// a SIMD, and in 160 KB of LDS a CU (taken in steps of 1280 bytes) what
// colour_lds gives, the tile's new snapshots and up to 512 bytes of counters.
// 1024 tiles of 16 x 32 cells with one layer, 768 with two; 768 and 512 near
// the widest halo.
inline int64_t colour_resident(const StepShape& sh, const ColourHalo& h, bool track, int32_t layers) {
  const int64_t lds = colour_lds(sh, h, track, layers) + 4 * (int64_t)(sh.sx + 2) * (sh.sy + 2) * layers + 512;
  const int64_t by_lds = 163840 / ((lds + 1279) / 1280 * 1280), by_waves = 16 / (sh.threads / 64);
  return 256 * (by_lds < by_waves ? by_lds : by_waves);
}

// Whether a window of the colour-ordered cascade runs as one launch
// (k_colour_step) or as a step launch and one launch per colour class.  Fused,
// a window costs its rounds of workgroups (tiles / resident), each running 3
// to 5 regions' cascades a tile; the classes cost `classes` launches, which
// past a few rounds fill the chip too.  So the line is a number of rounds that
// grows with the classes, and moves out where few cells are visited (a tile's
// cascades are then few) or, with one layer, nearly all are (their events
// shrink to the steep cells).  Measured, ms a 66-window cycle fused / classes:
// 1024^2 periodic (16 classes, 2.7 rounds), two layers, 0.25 particles a cell
// 10.8 / 12.3; 726^2 (9, 1.4) 6.9 / 6.9; 900^2 (9, 2.2) 9.4 / 8.6; 1025^2
// (25, 4.2) 15.8 / 15.8; 2048^2 (25, 16) 45.2 / 27.3; one layer there (10.7)
// 26.2 / 19.7, at one particle a cell 1281^2 (9, 3.2) 10.4 / 10.3; at 0.08
// 2050^2 (16, 10.9), two layers, 19.9 / 20.2; at 0.02 always fused up to 10
// rounds (2048^2, 16 rounds, 22.2 / 22.0).  Over 322 maps, densities and
// layers the choice costs 0.3% more than the better of the two.
inline bool colour_fused(int64_t tiles, int64_t resident, int32_t classes, int32_t layers, double per_cell) {
  double rounds;
  if (per_cell < 0.2) {
    rounds = classes * (0.04 + 0.04 / (per_cell > 0.033 ? per_cell : 0.033)) * (layers == 1 ? 1.3 : 1.0);
  } else if (layers == 1) {
    rounds = per_cell < 0.5 ? 0.225 * classes : 0.46 * classes;
    if (rounds > 10.0) rounds = 10.0;
  } else {
    rounds = 0.2 * classes - 0.5;
    if (rounds > 4.0) rounds = 4.0;
  }
  return (double)tiles <= rounds * (double)resident;
}

// One terrain of a context: its cells, tiles and particles are contiguous
// ranges of the context's buffers
struct Terrain {
  int64_t cell0;   // first cell in the map arrays
  int64_t part0;   // first particle index of a cycle
  int64_t npart;   // particles per cycle
  int32_t nx, ny, tiles_x, tiles_y, tile0;
  float rcp_nx, rcp_ny;
  uint64_t seed;
  float ps[3], nps[3];  // pspeed and normalize(pspeed)
};

// One particle record: 40 bytes (two 16-byte words and the ledger), moved
// with three vector loads or stores at immediate offsets from one address
// (8-byte aligned; global loads and stores of 16 bytes need only 4).  The
// number of calls a particle has made (its age) is the window index: every
// live particle makes one call per window from window 0.  A particle whose
// position left a bounded map (or stopped being finite) is stored with the
// bits of its last cell in q0.x and a NaN in q0.z: its next call finds no
// cell, and it dies (and deposits) at that cell.
typedef float f4a8 __attribute__((ext_vector_type(4), aligned(8)));
struct PRec {
  f4a8 q0;         // pos.xyz, sediment (off the map: last cell's bits, -, NaN, sediment)
  f4a8 q1;         // speed.xyz, particle index bits (RNG stream)
  int64_t ledger;  // fixed-point load
};
static_assert(sizeof(PRec) == 40 && alignof(PRec) == 8, "particle record: 40 bytes");

struct StepArgs {
  // map, window parity in -> out.  A master holds the previous window's
  // pickups already; its cascades are added here (relax), then this
  // window's pickups before it is written out.
  const int64_t* zm_in;
  int64_t* zm_out;
  const float* snap_in;  // snapshot the previous window's particles read
  float* snap_out;       // snapshot of this window (master after the relax)
  const int64_t* sm_in;
  int64_t* sm_out;
  const float* ssnap_in;
  float* ssnap_out;
  const uint32_t* v_in;  // previous window's cascade events
  uint32_t* v_out;
  int64_t* trk;          // 4 x ncell tracks of the cycle
  int64_t* lost;         // kLostSlots counters
  uint64_t* stat;        // kStatKinds x kStatSlots statistics
  // particles
  const PRec* in;
  PRec* out;
  const PRec* far_in;
  PRec* far_out;
  uint32_t* far_cnt_in;
  uint32_t* far_cnt_out;
  uint32_t* far_cnt_clear;   // the far counter of the window after next
  // routing: 9 sub-ranges (one per direction) of each tile's output region
  const int64_t* sub_base_prev;  // [tile * 9 + d] start of sub-range d in `in`
  const uint32_t* sub_cnt_prev;  // [tile * 9 + d] its length
  int64_t* sub_base_cur;         // the same for `out` (written here)
  uint32_t* sub_cnt_cur;
  const uint32_t* nin_cur;   // particles each tile receives this window
  uint32_t* nin_next;        // ... next window (accumulated here)
  uint32_t* nin_clear;       // ... the window after next (zeroed here)
  const uint32_t* csum_cur;  // nin_cur summed over chunks of kStepChunk tiles
  uint32_t* csum_next;
  uint32_t* csum_clear;
  const uint64_t* cycle;
  const Terrain* terr;
  const int32_t* tile_terrain;  // per global tile
  // 1: every tile is terrain t0 (no lookups).  A single map with the context's
  // seed and wind only: a captured cycle holds its arguments, and a terrain
  // with its own may change them from call to call.
  int32_t one_terrain;
  Terrain t0;
  int64_t ncell;                // cells of all terrains (track plane stride)
  int32_t ntiles;
  float mapscale, boundarylayer, suspension, gravity, abrasion, maxdiff, settling;
  int32_t max_age;
  // workgroup -> tile order: 0 = each XCD a contiguous range of tiles;
  // C >= 1 = runs of C consecutive tiles dealt round-robin over the XCDs
  int32_t tile_order;
  // crowded tiles first: a tile with more than kHeavyMin arrivals in one
  // window is listed for the next launch, whose first heavy_slots
  // workgroups take the listed tiles (so they start at once instead of
  // finishing last); the workgroup of the usual order then skips the tile
  int32_t heavy_slots;       // 0 = off, else a multiple of 8 (XCD mapping)
  int32_t default_slots;     // workgroups of the usual order: ntiles (a multiple of 8 with light slots)
  int32_t light_slots;       // 0 = off, else a multiple of 8: light tiles last, per XCD
  int32_t window;            // window index within the cycle
  ColourHalo chalo;          // colour-ordered relax: halo of tiles near a seam (the widest of all terrains)
  const uint32_t* heavy_cur; // this launch's listed tiles: kHeavySlotsMax heavy, then light_slots light,
                             // each part in 8 equal per-XCD lists
  uint32_t* heavy_next;      // the next launch's (appended here)
  const uint32_t* hcnt_cur;  // list lengths (may exceed the slots): [x] heavy, [8 + x] light on XCD x
  uint32_t* hcnt_next;
  uint32_t* hcnt_clear;      // the lengths of the lists after next
  uint32_t* hstamp;          // per tile: w + 1 when listed for window w (0 at cycle start)
};

#ifndef SWE_HEAVY_MIN
#define SWE_HEAVY_MIN 1024
#endif
#ifndef SWE_HEAVY_SLOTS
#define SWE_HEAVY_SLOTS 256
#endif
#ifndef SWE_LIGHT_MAX
#define SWE_LIGHT_MAX 256
#endif
constexpr uint32_t kHeavyMin = SWE_HEAVY_MIN;        // arrivals that make a tile heavy
constexpr uint32_t kLightMax = SWE_LIGHT_MAX;        // arrivals that leave a tile light
constexpr int32_t kHeavySlotsMax = SWE_HEAVY_SLOTS;  // listed tiles per launch (a multiple of 8)

struct SpawnArgs {
  PRec* out;
  int32_t* tile;     // per particle
  uint32_t* rank;    // per particle
  uint32_t* count;   // per tile, zero on entry: window 0's input counts
  uint32_t* csum;    // per chunk of kStepChunk tiles: window 0's chunk sums
  int64_t* sub_base; // [tile * 9 + d]: window 0's arrivals, all in d = 4 (own tile)
  uint32_t* sub_cnt;
  const uint64_t* cycle;
  const Terrain* terr;
  int32_t nterr;
  int64_t n;         // particles of all terrains
  int32_t ntiles;
  int32_t periodic, spawn_mode;
  int32_t tile_sx, tile_sy;  // the tile shape the particles are binned for
};

void launch_step(int shape, const StepArgs& a, bool periodic, bool track, int layers, bool deposit,
                 int mode, hipStream_t s);
#define SWE_DECLARE_SHAPE(i)                                                                                    \
  void launch_step_shape##i(const StepArgs& a, bool periodic, bool track, int layers, bool deposit, int mode, \
                            hipStream_t s);
SWE_DECLARE_SHAPE(0)
SWE_DECLARE_SHAPE(1)
SWE_DECLARE_SHAPE(2)
SWE_DECLARE_SHAPE(3)
SWE_DECLARE_SHAPE(4)
#undef SWE_DECLARE_SHAPE
void launch_spawn(const SpawnArgs& a, hipStream_t s);

}  // namespace swe
