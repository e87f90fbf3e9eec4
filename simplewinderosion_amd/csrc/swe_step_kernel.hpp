// swe_step_kernel.hpp -- the tile-owned step kernel for one-call snapshot
// windows, templated on the tile shape (SX x SY cells, NT threads, a
// register budget of WPE waves per SIMD); each shape is instantiated in its
// own translation unit (swe_step_shapes.hip).
//
// With window == 1 every fly() call writes only to the particle's pre-move
// cell, i.e. the cell it occupies when the window starts.  k_step gives each
// workgroup one tile of kSX x kSY cells and the particles currently in it,
// so all of a window's writes land in LDS of the owning workgroup and reach
// HBM as plain coalesced stores -- no global atomics.  One launch per window:
//
//   1. relax of the previous window (the k_relax stencil) for the tile plus
//      a one-cell halo, recomputed redundantly from a three-cell snapshot
//      halo in LDS: master/snapshot of the tile written out, the halo kept in
//      LDS for the particles' five-point stencils;
//   2. one fly() call (wind.hpp:28-117) for every particle in the tile
//      against the LDS snapshot; pickups, cascade-event counts and tracks
//      summed in LDS (int64 / uint32) and stored once per cell;
//   3. routing: the tile's output region of the particle buffer has nine
//      sub-ranges, one per direction (-1, 0, +1)^2 of the tile a particle now
//      occupies, each with room for all the tile's particles; a particle is
//      appended to the sub-range of its direction.  The per-direction counts
//      are added to the destination tiles' input counts for the next window
//      (and to the sums of chunks of kChunk tiles), from which every
//      workgroup derives the start of its own output region.  A tile reads
//      its arrivals from the nine sub-ranges that point at it: no scan.
//
// A particle that jumps more than one tile (never seen in practice) goes to a
// "far" list that every workgroup scans for particles in its tile.
#pragma once

#include "swe_cascade.hpp"
#include "swe_fly.hpp"
#include "swe_kernels.h"
#include "swe_step.h"

namespace swe {

constexpr int kChunk = kStepChunk;   // tiles per input-count chunk sum
constexpr uint32_t kCrowded = 2048;  // tile load counted as crowded in the statistics

constexpr int32_t c_ox[8] = {-1, -1, -1, 0, 0, 1, 1, 1};
constexpr int32_t c_oy[8] = {-1, 0, 1, -1, 1, -1, 0, 1};

// LDS-backed stencil and accumulator for one tile (kH1Y: row length of the
// one-cell halo, kCell: cells of the tile)
template <int kH1Y>
struct TileMap {
  const float* s_new;   // H1 heights
  const float* s_snew;  // H1 sediment
  int32_t c;            // H1 index of the particle's cell
  __device__ float h(int dx, int dy) const { return s_new[c + dx * kH1Y + dy]; }
  __device__ float s0() const { return s_snew[c]; }
};

template <int kCell>
struct TileAcc {
  int64_t* d;
  int64_t* ds;
  uint32_t* v;
  int64_t* t;
  int32_t li;  // tile-local index of the particle's cell
  __device__ void add_pickup(int64_t, int64_t q, bool both) {
    atomicAdd((unsigned long long*)&d[li], (unsigned long long)q);
    if (both) atomicAdd((unsigned long long*)&ds[li], (unsigned long long)q);
  }
  __device__ void add_event(int64_t) { atomicAdd(&v[li], 1u); }
  __device__ void add_track(int64_t, float sed, f3 sp) {
    atomicAdd((unsigned long long*)&t[li], (unsigned long long)fx_from_f32(sed));
    atomicAdd((unsigned long long*)&t[kCell + li], (unsigned long long)fx_from_f32(sp.x));
    atomicAdd((unsigned long long*)&t[2 * kCell + li], (unsigned long long)fx_from_f32(sp.y));
    atomicAdd((unsigned long long*)&t[3 * kCell + li], (unsigned long long)fx_from_f32(sp.z));
  }
};

extern __shared__ __attribute__((aligned(16))) unsigned char s_dyn[];  // k_colour_step's working sets

__device__ __forceinline__ int32_t wrapt(int32_t v, int32_t n) {
  // small-range wrap for tile coordinates (|v| < 2n)
  if (v < 0) v += n;
  if (v >= n) v -= n;
  return v;
}

// The kernel's arguments, read where they are used: they exceed the scalar
// registers, and a value loaded at the start and held through the particle
// loop would be spilled to vector lanes and come back by v_readlane.  Each
// phase takes the pointer through step_args, which the compiler cannot see
// through, so its loads are not moved above it.
typedef const __attribute__((address_space(4))) StepArgs* StepArgsPtr;
typedef const __attribute__((address_space(4))) Terrain* TerrainPtr;
__device__ __forceinline__ StepArgsPtr step_args(StepArgsPtr p) {
  asm volatile("" : "+s"(p));
  return p;
}

// the register budget keeps WPE waves per SIMD (the default shape: five, and
// with the LDS of one workgroup under 32 KiB five workgroups share a CU)
// MODE 0: relax of the previous window (synchronous cascade) + one fly()
// call per particle; MODE 1: the relax only (the cycle's last window);
// MODE 2: the fly() calls only -- the previous window was relaxed before the
// launch by the colour-ordered cascade (one launch per colour class, on maps
// under three cells along an axis and where colour_fused prefers it), so the
// tile reads the snapshot and masters as they are.
// MODE 3, 4 (k_colour_step below): as 0 and 1 with the colour-ordered
// cascade run inside the tile.
template <int SX, int SY, int NT, bool PERIODIC, bool TRACK, int LAYERS, bool DEPOSIT, int MODE>
__device__ __forceinline__ void step_body() {
  StepArgsPtr ap = step_args((StepArgsPtr)__builtin_amdgcn_kernarg_segment_ptr());
  constexpr bool RELAX_ONLY = MODE == 1 || MODE == 4, EXT = MODE == 2, COLOUR = MODE >= 3;
  constexpr int kSX = SX, kSY = SY;
  constexpr int kH3X = kSX + 6, kH3Y = kSY + 6;  // snapshot halo 3
  constexpr int kH2X = kSX + 4, kH2Y = kSY + 4;  // events halo 2
  constexpr int kH1X = kSX + 2, kH1Y = kSY + 2;  // new values halo 1
  constexpr int kStepThreads = NT;
  constexpr int kCell = kSX * kSY;
  __shared__ float s_new[kH1X * kH1Y];
  __shared__ float s_snew[LAYERS == 2 ? kH1X * kH1Y : 1];
  // relax-phase and march-phase working sets share one buffer
  constexpr int kRelaxBytes =
      4 * kH3X * kH3Y * (LAYERS == 2 ? 2 : 1) + 4 * kH2X * kH2Y + 8 * kH1X * kH1Y * (LAYERS == 2 ? 2 : 1) + 2 * kH2X * kH2Y;
  constexpr int kMarchBytes = 8 * kCell * (LAYERS == 2 ? 2 : 1) + 4 * kCell + (TRACK ? 32 * kCell : 0);
  constexpr int kWorkBytes = kRelaxBytes > kMarchBytes ? kRelaxBytes : kMarchBytes;
  __shared__ __attribute__((aligned(16))) unsigned char s_static[COLOUR ? 16 : kWorkBytes];
  unsigned char* s_work = COLOUR ? s_dyn : s_static;
  __shared__ uint32_t s_slot[9];     // particles sent in direction d
  __shared__ int64_t s_rbase[9];     // arrivals: sub-range d of the source tile
  __shared__ uint32_t s_rpre[10];    // exclusive prefix of the sub-range lengths
  __shared__ int64_t s_part[kStepThreads / 64];
  __shared__ int64_t s_lost;         // load of the particles that died here
  __shared__ uint32_t s_far;         // particles that skipped a tile
  __shared__ int64_t s_base;
  __shared__ uint32_t s_ncas;        // cells whose cascade moves material
  __shared__ uint32_t s_ccnt[COLOUR ? 32 : 1];  // visited cells per colour class
  __shared__ uint32_t s_cpre[COLOUR ? 33 : 1];  // exclusive prefix of s_ccnt
  __shared__ uint32_t s_nready[2];              // cells listed in a round (by parity)
  __shared__ uint32_t s_large;                  // the region holds a master of 2^39 or more

  // XCD-aware order (workgroup b runs on XCD b % 8).  tile_order 0: XCD k
  // takes a contiguous range of tiles, so neighbouring tiles share halo
  // lines in one L2.  tile_order C >= 1: runs of C consecutive tiles are
  // dealt round-robin over the XCDs (evens out crowded regions); the last
  // nb mod 8C workgroups keep their own index.  Both are bijections.
  // The first heavy_slots workgroups take the tiles listed as crowded by the
  // previous launch, the last light_slots ones the tiles listed as light
  // (at most kLightMax arrivals), both listed per home XCD (the XCD that
  // takes the tile in the usual order), so a listed tile keeps its L2;
  // empty slots return at once.  The rest follow the usual order and skip
  // a listed tile.  heavy_slots and default_slots (with light slots) are
  // multiples of 8, so slot b of each part runs on XCD b % 8.
  const uint32_t hs = RELAX_ONLY ? 0u : (uint32_t)ap->heavy_slots;
  const uint32_t ls = RELAX_ONLY ? 0u : (uint32_t)ap->light_slots;
  const uint32_t nb = (uint32_t)ap->default_slots, b = blockIdx.x - (uint32_t)ap->heavy_slots;
  const uint32_t xcd = b % 8;
  int32_t u;  // global tile
  bool listed = false;
  if (blockIdx.x < (uint32_t)ap->heavy_slots) {
    const uint32_t k = blockIdx.x / 8;  // heavy slot k of this XCD (blockIdx.x % 8 == xcd)
    if (hs == 0) return;
    // the list entry is read together with the list length (k < hs / 8, so
    // it lies inside the list whatever the length; unused when k >= length)
    const uint32_t cnt = ap->hcnt_cur[xcd];
    const uint32_t cand = ap->heavy_cur[xcd * (hs / 8) + k];
    if (k >= cnt) return;
    u = (int32_t)cand;
    listed = true;
  } else if (b >= nb) {
    const uint32_t bl = b - nb, k = bl / 8;  // k < ls / 8
    if (ls == 0) return;
    const uint32_t cnt = ap->hcnt_cur[8 + xcd];
    const uint32_t cand = ap->heavy_cur[kHeavySlotsMax + xcd * (ls / 8) + k];
    if (k >= cnt) return;
    u = (int32_t)cand;
    listed = true;
  } else if (ap->tile_order <= 0) {
    const uint32_t q8 = nb / 8, r8 = nb % 8;
    u = (int32_t)(xcd * q8 + (xcd < r8 ? xcd : r8) + b / 8);
  } else {
    const uint32_t C = (uint32_t)ap->tile_order, full = nb / (8 * C) * (8 * C), j = b / 8;
    u = b < full ? (int32_t)(((j / C) * 8 + xcd) * C + j % C) : (int32_t)b;
  }
  if (u >= ap->ntiles) return;  // padding of the usual order to a multiple of 8
  // home XCD of tile t in the usual order: the XCD whose workgroups take it
  auto home_of = [&](uint32_t t) __attribute__((always_inline)) -> uint32_t {
    if (ap->tile_order <= 0) {
      const uint32_t q8 = nb / 8, r8 = nb % 8;
      return t < r8 * (q8 + 1) ? t / (q8 + 1) : r8 + (t - r8 * (q8 + 1)) / q8;
    }
    const uint32_t C = (uint32_t)ap->tile_order, full = nb / (8 * C) * (8 * C);
    return t < full ? (t / C) % 8 : t % 8;
  };
  // a listed tile's stamp is window + 1 (or window + 2 once its listed
  // workgroup has listed it again): either way the usual one skips it,
  // before it loads anything
  if ((hs | ls) > 0 && !listed && ap->hstamp[u] > (uint32_t)ap->window) return;
  // the terrain this tile belongs to; all map indices below are terrain-local
  // (a single map's record is among the arguments: no dependent load there)
  TerrainPtr tp = &ap->t0;
  if (!ap->one_terrain) tp = (TerrainPtr)(uintptr_t)(ap->terr + ap->tile_terrain[u]);
  const int32_t nx = tp->nx, ny = tp->ny;
  const int32_t tiles_x = tp->tiles_x, tiles_y = tp->tiles_y;
  const int32_t t0 = tp->tile0;
  const int32_t ul = u - t0;
  const int32_t tx = ul / tiles_y, ty = ul % tiles_y;
  const int32_t x0 = tx * kSX, y0 = ty * kSY;
  const float rcp_nx = tp->rcp_nx, rcp_ny = tp->rcp_ny;
  const int64_t c0 = tp->cell0;
  const int64_t* zm_in = ap->zm_in + c0;
  const float* snap_in = ap->snap_in + c0;
  float* snap_out = ap->snap_out + c0;
  const int64_t* sm_in = LAYERS == 2 ? ap->sm_in + c0 : nullptr;
  const float* ssnap_in = LAYERS == 2 ? ap->ssnap_in + c0 : nullptr;
  float* ssnap_out = LAYERS == 2 ? ap->ssnap_out + c0 : nullptr;
  const uint32_t* v_in = ap->v_in + c0;
  // a halo coordinate's wrap: within one period on an axis of 64 cells or
  // more (the halo is at most 31 cells, the last tile's overhang 31)
  auto wrap_x = [&](int32_t v) __attribute__((always_inline)) {
    return nx >= 64 ? wrap_near(v, nx) : wrap(v, nx, rcp_nx);
  };
  auto wrap_y = [&](int32_t v) __attribute__((always_inline)) {
    return ny >= 64 ? wrap_near(v, ny) : wrap(v, ny, rcp_ny);
  };

  constexpr int kCellPer = (kCell + kStepThreads - 1) / kStepThreads;

  // this window's output region starts at 9 x (input counts of tiles 0 ..
  // u-1): the chunk sums of the earlier chunks plus the earlier tiles of this
  // chunk.  The loads are issued here and summed after the relax phase (no
  // wait on them before the map loads go out).
  static_assert(kChunk <= kStepThreads, "one tile of the current chunk per thread");
  uint32_t part_c = 0, part_n = 0;
  {
    const int32_t cu = u / kChunk;
    if (cu <= kStepThreads) {
      if ((int32_t)threadIdx.x < cu) part_c = ap->csum_cur[threadIdx.x];
    } else {
      for (int32_t c = threadIdx.x; c < cu; c += kStepThreads) part_c += ap->csum_cur[c];
    }
    const int32_t t = cu * kChunk + (int32_t)threadIdx.x;
    if (t < u) part_n = ap->nin_cur[t];
  }
  const uint32_t nin_u = RELAX_ONLY ? 0u : ap->nin_cur[u];
  // read here, so that the particle phase does not start by waiting for them
  const uint64_t cycle = RELAX_ONLY ? 0u : *ap->cycle;
  const uint32_t far_n = RELAX_ONLY ? 0u : *ap->far_cnt_in;

  PRec rec0{};       // this thread's first arrival (loaded in the relax phase)
  uint32_t sr0 = 0;  // its sub-range
  // arrivals of this window: the source tile in direction -d of this one
  // wrote the particles that moved by d into its sub-range d
  auto load_arrivals = [&]() __attribute__((always_inline)) {
    if (threadIdx.x < 9) {
      const int32_t d = threadIdx.x, dx = d / 3 - 1, dy = d % 3 - 1;
      int32_t sx = tx - dx, sy = ty - dy;
      bool ok = !RELAX_ONLY;
      if (PERIODIC) {
        sx = wrapt(sx, tiles_x);
        sy = wrapt(sy, tiles_y);
      } else {
        ok = ok && sx >= 0 && sy >= 0 && sx < tiles_x && sy < tiles_y;
      }
      int64_t rb = 0;
      uint32_t rc = 0;
      if (ok) {
        const int64_t s9 = (int64_t)(t0 + sx * tiles_y + sy) * 9 + d;
        rb = ap->sub_base_prev[s9];
        rc = ap->sub_cnt_prev[s9];
      }
      s_rbase[d] = rb;
      s_slot[d] = rc;  // lengths, turned into s_rpre by prefix_arrivals
    }
  };
  auto prefix_arrivals = [&]() __attribute__((always_inline)) {
    if (threadIdx.x == 0) {
      uint32_t r = 0;
      for (int d = 0; d < 9; d++) {
        s_rpre[d] = r;
        r += s_slot[d];
      }
      s_rpre[9] = r;
    }
  };
  auto first_arrival = [&]() __attribute__((always_inline)) {
    if (threadIdx.x < s_rpre[9]) {
      while (sr0 < 8 && threadIdx.x >= s_rpre[sr0 + 1]) sr0++;
      rec0 = ap->in[s_rbase[sr0] + (int64_t)(threadIdx.x - s_rpre[sr0])];
    }
  };
  if constexpr (EXT) {
    // ---------------- 1'. the relaxed map of the previous window ----------------
    // one-halo snapshot into LDS for the particles' stencils, the tile's
    // masters into the pickup accumulators; all loads issued first
    constexpr int kH1Per = (kH1X * kH1Y + kStepThreads - 1) / kStepThreads;
    float hv[kH1Per], hs1[LAYERS == 2 ? kH1Per : 1];
    int64_t zt[kCellPer], st[LAYERS == 2 ? kCellPer : 1];
#pragma unroll
    for (int i = 0; i < kH1Per; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      int32_t gx = x0 - 1 + e / kH1Y, gy = y0 - 1 + e % kH1Y;
      bool ok = e < kH1X * kH1Y;
      if (PERIODIC) {
        gx = wrap_x(gx);
        gy = wrap_y(gy);
      } else {
        ok = ok && gx >= 0 && gy >= 0 && gx < nx && gy < ny;
      }
      const int64_t g = (int64_t)gx * ny + gy;
      hv[i] = ok ? snap_in[g] : 0.0f;
      if (LAYERS == 2) hs1[i] = ok ? ssnap_in[g] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kCellPer; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      const int32_t gx = x0 + e / kSY, gy = y0 + e % kSY;
      const bool ok = e < kCell && gx < nx && gy < ny;
      const int64_t g = (int64_t)gx * ny + gy;
      zt[i] = ok ? zm_in[g] : 0;
      if (LAYERS == 2) st[i] = ok ? sm_in[g] : 0;
    }
    load_arrivals();
    int64_t* acc_z = (int64_t*)s_work;
#pragma unroll
    for (int i = 0; i < kH1Per; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      if (e < kH1X * kH1Y) {
        s_new[e] = hv[i];
        if (LAYERS == 2) s_snew[e] = hs1[i];
      }
    }
#pragma unroll
    for (int i = 0; i < kCellPer; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      if (e < kCell) {
        acc_z[e] = zt[i];
        if (LAYERS == 2) acc_z[kCell + e] = st[i];
      }
    }
    __syncthreads();
    prefix_arrivals();
    __syncthreads();
    first_arrival();
  } else if constexpr (COLOUR) {
  // ---------------- 1''. colour-ordered relax of the previous window ----------------
  // The masters (with the previous window's pickups) of the tile and the
  // halo its result depends on, in LDS; every visited cell's cascade there
  // runs on them in class order.
  {
    // a tile whose widest halo meets a cell of the classes past 2 (the last
    // n mod 3 cells of a periodic axis) takes that halo, any other the
    // interior one (swe_step.h: kColourHalo, colour_halo)
    ColourHalo hl = kColourHalo;
    const int32_t limx = PERIODIC ? nx - nx % 3 : nx, limy = PERIODIC ? ny - ny % 3 : ny;
    if (PERIODIC) {
      const ColourHalo w = {ap->chalo.xl, ap->chalo.xh, ap->chalo.yl, ap->chalo.yh};
      const bool sx = limx != nx && (x0 - w.xl < 0 || x0 + kSX + w.xh > limx);
      const bool sy = limy != ny && (y0 - w.yl < 0 || y0 + kSY + w.yh > limy);
      if (sx || sy) hl = w;
    }
    const int32_t RX = kSX + hl.xl + hl.xh, RY = kSY + hl.yl + hl.yh, R = RX * RY;
    const float rcp_ry = 1.0f / (float)RY;
    int64_t* z_r = (int64_t*)s_work;
    int64_t* s_r = z_r + R;  // LAYERS == 2
    uint32_t* v_r = (uint32_t*)(z_r + R * LAYERS);
    uint16_t* list = (uint16_t*)(v_r + R);
    // class of a visited cell whose cascade has not run yet (1 ..), else 0;
    // a row and eight cells of zeros before and after it, so that the 5 x 5
    // neighbourhood of any listed cell can be read in eight-byte rows
    uint8_t* cls = (uint8_t*)(list + R) + RY + 8;
    if (threadIdx.x < 32) s_ccnt[threadIdx.x] = 0;
    if (threadIdx.x < 2) s_nready[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_large = 0;
    for (int32_t e = threadIdx.x; e < RY + 8; e += kStepThreads) {
      cls[e - RY - 8] = 0;
      cls[R + e] = 0;
    }
    // region row of index e (e < 2^16: the product is within 1/2 of a step of exact)
    auto row_of = [=](int32_t e) __attribute__((always_inline)) {
      return (int32_t)(((float)e + 0.5f) * rcp_ry);
    };
    // A wave loads whole rows, 64 columns at a time (the interior region is 62
    // wide): the row's address and x class are scalar, the column's part is
    // computed once.
    constexpr int kWaves = kStepThreads / 64;
    constexpr int kRows = (kSX + kColourHaloMax.xl + kColourHaloMax.xh + kWaves - 1) / kWaves;
    constexpr int kChunks = (kSY + kColourHaloMax.yl + kColourHaloMax.yh + 63) / 64;
    // rows a wave has in flight (eight overflow the registers of the closing
    // launch of the largest shape)
    constexpr int kMost = RELAX_ONLY && kStepThreads > 256 ? 4 : 8, kB = kRows < kMost ? kRows : kMost;
    const int32_t wv = __builtin_amdgcn_readfirstlane((int32_t)threadIdx.x >> 6), lane = (int32_t)threadIdx.x & 63;
    uint32_t where[kChunks][kRows];  // class << 16 | rank in the wave's part of it; 0: not listed
    uint32_t wcnt = 0;
    bool large = false;  // a master the quick conversion below cannot take
    __syncthreads();
#pragma unroll
    for (int cc = 0; cc < kChunks; cc++) {
#pragma unroll
      for (int i = 0; i < kRows; i++) where[cc][i] = 0;
      if (64 * cc >= RY) continue;
      const int32_t ly = 64 * cc + lane;
      int32_t gy = y0 - hl.yl + ly;
      bool okc = ly < RY;
      if (PERIODIC) gy = wrap_y(gy);
      else okc = okc && gy >= 0 && gy < ny;
      const int32_t ccy = gy < limy ? gy % 3 : 3 + gy - limy;
      // the outermost ring only lends its values
      const bool okl = okc && ly >= 1 && ly < RY - 1;
#pragma unroll
      for (int b0 = 0; b0 < kRows; b0 += kB) {
        int64_t zv[kB], sv[LAYERS == 2 ? kB : 1];
        uint32_t vv[kB];
#pragma unroll
        for (int j = 0; j < kB; j++) {
          const int32_t lx = wv + (b0 + j) * kWaves;
          zv[j] = 0;
          if (LAYERS == 2) sv[j] = 0;
          vv[j] = 0;
          int32_t gx = x0 - hl.xl + lx;
          bool okr = b0 + j < kRows && lx < RX;
          if (PERIODIC) gx = wrap_x(gx);
          else okr = okr && gx >= 0 && gx < nx;
          if (!okr) continue;
          const int64_t g = (int64_t)gx * ny + gy;
          if (okc) {
            zv[j] = zm_in[g];
            if (LAYERS == 2) sv[j] = sm_in[g];
          }
          if (okl && lx >= 1 && lx < RX - 1) vv[j] = v_in[g];
        }
        if (cc == 0 && b0 == 0) load_arrivals();
#pragma unroll
        for (int j = 0; j < kB; j++) {
          const int32_t lx = wv + (b0 + j) * kWaves;
          if (b0 + j >= kRows || lx >= RX) continue;
          int32_t gx = x0 - hl.xl + lx;
          if (PERIODIC) gx = wrap_x(gx);
          const int32_t cv = (gx < limx ? gx % 3 : 3 + gx - limx) * kColourAxisMax + ccy + 1;
          const int32_t e = lx * RY + ly;
          const bool act = vv[j] != 0;
          if (ly < RY) {
            z_r[e] = zv[j];
            if (LAYERS == 2) s_r[e] = sv[j];
            v_r[e] = vv[j];
            large = large || !small_fx(zv[j]) || (LAYERS == 2 && !small_fx(sv[j]));
            cls[e] = (uint8_t)(act ? cv : 0);
          }
          // rank within the wave's cells of the class (lane c of wcnt counts class c)
          uint64_t rem = __ballot(act);
          while (rem) {
            const int32_t c = __builtin_amdgcn_readlane(cv, __builtin_ctzll(rem));
            const bool in = act && cv == c;
            const uint64_t m = __ballot(in);
            const uint32_t base = __builtin_amdgcn_readlane(wcnt, c);
            const uint32_t below =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (in) where[cc][b0 + j] = (uint32_t)c << 16 | (base + below);
            if (lane == c) wcnt += (uint32_t)__popcll(m);
            rem &= ~m;
          }
        }
      }
    }
    // this wave's part of each class's list starts at wcnt
    if (lane < 32) wcnt = wcnt ? atomicAdd(&s_ccnt[lane], wcnt) : 0u;
    if (__ballot(large) && lane == 0) s_large = 1;
    __syncthreads();
    prefix_arrivals();
    if (threadIdx.x >= kStepThreads - 64) {  // the last wave: prefix over the classes
      const int32_t l = (int32_t)threadIdx.x & 63;
      const uint32_t v = l < 32 ? s_ccnt[l] : 0u;
      uint32_t t = v;
#pragma unroll
      for (int off = 1; off < 32; off <<= 1) {
        const uint32_t y = __shfl_up(t, off, 64);
        if (l >= off) t += y;
      }
      if (l < 32) s_cpre[l] = t - v;
      if (l == 31) s_cpre[32] = t;
    }
    __syncthreads();
#pragma unroll
    for (int cc = 0; cc < kChunks; cc++)
#pragma unroll
      for (int i = 0; i < kRows; i++)
        if (__ballot(where[cc][i] != 0)) {
          const uint32_t w = where[cc][i], base = __shfl(wcnt, (int)(w >> 16), 64);
          if (w)
            list[s_cpre[w >> 16] + base + (w & 0xffffu)] = (uint16_t)((wv + i * kWaves) * RY + 64 * cc + lane);
        }
    const uint32_t nvis = s_cpre[32];
    if (!RELAX_ONLY) first_arrival();
    __syncthreads();

    // Masters below 2^39 at the start (heights below 128) stay below 2^47
    // through the relax: with settling in [0, 1] and a threshold of zero or
    // more a transfer is at most half the difference of the two heights, so
    // heights stay within the region's range, and a cell's sediment sees at
    // most 8 x 25 transfers.  Those take the short conversion.
    const bool quick =
        s_large == 0 && ap->settling >= 0.0f && ap->settling <= 1.0f && ap->maxdiff >= 0.0f;
    // one cell's cascade on the LDS masters
    auto relax = [&](int32_t e) __attribute__((always_inline)) {
      const int32_t lx = row_of(e), ly = e - lx * RY;
      const int32_t gx = x0 - hl.xl + lx, gy = y0 - hl.yl + ly;
      int64_t zn[8];
#pragma unroll
      for (int k = 0; k < 8; k++) zn[k] = z_r[e + c_ox[k] * RY + c_oy[k]];
      const int64_t zc = z_r[e];
      float hc = f32_from_small_fx(zc);
      float hn[8];
#pragma unroll
      for (int k = 0; k < 8; k++) hn[k] = f32_from_small_fx(zn[k]);
      if (!quick) {
        hc = f32_from_fx(zc);
#pragma unroll
        for (int k = 0; k < 8; k++) hn[k] = f32_from_fx(zn[k]);
      }
      uint32_t valid = 0;
      // no neighbour beyond the threshold: the walk moves nothing
      float most = -1.0f;
      const float dd = __builtin_sqrtf(2.0f);
#pragma unroll
      for (int k = 0; k < 8; k++) {
        bool ok = true;
        if (!PERIODIC) {
          const int32_t qx = gx + c_ox[k], qy = gy + c_oy[k];
          ok = qx >= 0 && qy >= 0 && qx < nx && qy < ny;
        }
        valid |= (ok ? 1u : 0u) << k;
        const float ad = __builtin_fabsf(hc - hn[k]);
        const float d = (c_ox[k] != 0 && c_oy[k] != 0) ? dd : 1.0f;
        const float m = __builtin_fminf(ad - (d * ap->maxdiff) * 1.0f, ad);
        most = __builtin_fmaxf(most, ok ? m : -1.0f);
      }
      if (!(most > 0.0f)) return;
      const auto sed_at = [&](int32_t q) __attribute__((always_inline)) {
        const int64_t m = s_r[q];
        float f = f32_from_small_fx(m);
        if (!quick) f = f32_from_fx(m);
        return f;
      };
      const auto sed_of = [&](int32_t k) { return sed_at(e + off_x(k) * RY + off_y(k)); };
      int64_t centre = 0;
      cascade_cell_dev<LAYERS>(hn, sed_of, hc, LAYERS == 2 ? sed_at(e) : 0.0f, valid,
                               u2f(v_r[e]), ap->maxdiff, [&](int32_t k, int64_t amt) {
                                 centre -= amt;
                                 const int32_t q = e + off_x(k) * RY + off_y(k);
                                 // no other cell in flight touches q: the atomics only save the reads' wait
                                 if (amt != 0) {
                                   atomicAdd((unsigned long long*)&z_r[q], (unsigned long long)amt);
                                   if (LAYERS == 2) atomicAdd((unsigned long long*)&s_r[q], (unsigned long long)amt);
                                 }
                               });
      atomicAdd((unsigned long long*)&z_r[e], (unsigned long long)centre);
      if (LAYERS == 2) atomicAdd((unsigned long long*)&s_r[e], (unsigned long long)centre);
    };
    // Up to two visited cells a thread: in rounds, every cell that no visited
    // cell of an earlier class within two cells still precedes is listed
    // (cells further apart share no neighbour, and of two closer ones the
    // earlier class goes first), and the listed cells run on packed waves.
    // Dependences run down the classes, so there are at most as many rounds as
    // classes; scattered cells need two or three.  More cells: one class after
    // another.
    constexpr int kClasses = kColourAxisMax * kColourAxisMax;
    const bool few = nvis <= 2u * kStepThreads;
    const bool have0 = threadIdx.x < nvis, have1 = threadIdx.x + kStepThreads < nvis;
    const int32_t own0 = few && have0 ? list[threadIdx.x] : 0;
    const int32_t own1 = few && have1 ? list[threadIdx.x + kStepThreads] : 0;
    uint32_t pend = few ? (have0 ? 1u : 0u) | (have1 ? 2u : 0u) : 0u;
    uint32_t done = 0;
    // the visited cells' settling factors, in place of their events
    for (uint32_t i = threadIdx.x; i < nvis; i += kStepThreads) {
      const int32_t e = list[i];
      v_r[e] = f2u(settle_factor_dev(ap->settling, v_r[e]));
    }
    __syncthreads();  // (the list is in registers too: its storage takes the rounds' cells)
    for (int32_t round = 0; round < kClasses; round++) {
      const uint16_t* run = list;
      uint32_t n;
      if (few) {
        for (int q = 0; q < 2; q++) {
          bool ready = false;
          const int32_t e = q == 0 ? own0 : own1;
          if (pend & (1u << q)) {
            // the five rows of its neighbourhood, five cells each: no byte o
            // with 0 < o < mine (bytes are below 128, so per-byte sums and
            // differences do not carry)
            const uint8_t* p = cls + e - 2;
            const uint32_t mine = p[2] * 0x01010101u;
            uint32_t w[5], x[5];
#pragma unroll
            for (int dx = 0; dx < 5; dx++) {
              __builtin_memcpy(&w[dx], p + (dx - 2) * RY, 4);
              x[dx] = p[(dx - 2) * RY + 4];
            }
            const uint32_t xs = x[0] | x[1] << 8 | x[3] << 16 | x[4] << 24;
            uint32_t before = 0;
#pragma unroll
            for (int i = 0; i < 7; i++) {
              const uint32_t o = i < 5 ? w[i] : (i == 5 ? xs : x[2]);
              before |= ~((o | 0x80808080u) - mine) & (o + 0x7f7f7f7fu);
            }
            ready = (before & 0x80808080u) == 0;
          }
          const uint64_t m = __ballot(ready);
          if (m) {
            const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(&s_nready[round & 1], (uint32_t)__popcll(m));
            base = __builtin_amdgcn_readfirstlane(base);
            if (ready) {
              list[base + below] = (uint16_t)e;
              pend &= ~(1u << q);
            }
          }
          if (nvis <= (uint32_t)kStepThreads) break;
        }
        __syncthreads();
        n = s_nready[round & 1];
        if (threadIdx.x == 0) s_nready[(round & 1) ^ 1] = 0;
      } else {
        n = s_ccnt[round + 1];
        if (n == 0) continue;
        run = list + s_cpre[round + 1];
      }
      for (uint32_t i = threadIdx.x; i < n; i += kStepThreads) {
        const int32_t e = run[i];
        relax(e);
        cls[e] = 0;
      }
      __syncthreads();
      done += n;
      if (done >= nvis) break;
    }

    // the relaxed masters of the tile and its one-cell halo; the sediment
    // layer clamped at zero after the last class
    constexpr int kH1Per = (kH1X * kH1Y + kStepThreads - 1) / kStepThreads;
    int64_t zt[kH1Per], st[LAYERS == 2 ? kH1Per : 1];
#pragma unroll
    for (int i = 0; i < kH1Per; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      zt[i] = 0;
      if (LAYERS == 2) st[i] = 0;
      if (e >= kH1X * kH1Y) continue;
      const int32_t q = (hl.xl - 1 + e / kH1Y) * RY + hl.yl - 1 + e % kH1Y;
      zt[i] = z_r[q];
      if (LAYERS == 2) st[i] = s_r[q] < 0 ? 0 : s_r[q];
    }
    __syncthreads();
    int64_t* acc_z = (int64_t*)s_work;
#pragma unroll
    for (int i = 0; i < kH1Per; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      if (e >= kH1X * kH1Y) continue;
      const int32_t lx = e / kH1Y, ly = e % kH1Y;
      const float zf = f32_from_fx(zt[i]);
      s_new[e] = zf;  // cells off a bounded map hold 0
      const bool mine = lx >= 1 && ly >= 1 && lx <= kSX && ly <= kSY;
      const int32_t gx = x0 - 1 + lx, gy = y0 - 1 + ly, li = (lx - 1) * kSY + (ly - 1);
      const bool on = mine && gx < nx && gy < ny;
      const int64_t g = (int64_t)gx * ny + gy;
      if (mine) acc_z[li] = zt[i];
      if (RELAX_ONLY && on) snap_out[g] = zf;  // the cycle's last window leaves the snapshot
      if (LAYERS == 2) {
        const float sf = f32_from_fx(st[i]);
        s_snew[e] = sf;
        if (mine) acc_z[kCell + li] = st[i];
        if (RELAX_ONLY && on) ssnap_out[g] = sf;
      }
    }
    __syncthreads();
  }
  } else {
  // ---------------- 1. relax of the previous window ----------------
  {
    float* s_old = (float*)s_work;
    float* s_sold = s_old + kH3X * kH3Y;  // valid when LAYERS == 2
    uint32_t* s_vold = (uint32_t*)(s_old + kH3X * kH3Y * (LAYERS == 2 ? 2 : 1));
    // the 1-halo masters, to which the cascades' transfers are added; with two
    // layers also sediment minus height master, which a transfer leaves alone
    int64_t* s_casc = (int64_t*)(s_vold + kH2X * kH2Y);
    int64_t* s_sdif = s_casc + kH1X * kH1Y;  // LAYERS == 2
    // Cells of the halo region by thread: kPass passes of whole rows (a thread
    // keeps its column, kRPP rows a pass), then the six halo columns.  One
    // address serves a cell's five arrays (snapshot and sediment snapshot on
    // the 3-halo, events on the 2-halo, the masters with the previous window's
    // pickups on the 1-halo), and every load is issued before the first LDS
    // store, so the fill costs one memory round trip.  (Linear indices into
    // each region cost a division and a wrap per load: a sixth of the
    // kernel's vector instructions.)
    constexpr int kRPP = kStepThreads / kSY;
    constexpr int kPass = (kH3X + kRPP - 1) / kRPP;
    constexpr int kHaloCells = 6 * kH3X;
    constexpr int kItems = kPass + (kHaloCells + kStepThreads - 1) / kStepThreads;
    static_assert(kStepThreads % kSY == 0, "whole rows a pass");
    const int32_t trow = (int32_t)threadIdx.x / kSY, tcol = (int32_t)threadIdx.x % kSY + 3;
    // row and column of item i in the 3-halo region; false past its end
    auto item = [&](int i, int32_t& row, int32_t& col) __attribute__((always_inline)) {
      if (i < kPass) {
        row = trow + i * kRPP;
        col = tcol;
        return row < kH3X;
      }
      const int32_t h = (int32_t)threadIdx.x + (i - kPass) * kStepThreads;
      row = h / 6;
      const int32_t c = h - row * 6;
      col = c < 3 ? c : kSY + c;
      return h < kHaloCells;
    };
    float hv[kItems], hs3[LAYERS == 2 ? kItems : 1];
    uint32_t vv[kItems];
    int64_t zv[kItems], sv[LAYERS == 2 ? kItems : 1];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      int32_t row, col;
      bool ok = item(i, row, col);
      int32_t gx = x0 - 3 + row, gy = y0 - 3 + col;
      if (PERIODIC) {
        gx = wrap_x(gx);
        gy = wrap_y(gy);
      } else {
        ok = ok && gx >= 0 && gy >= 0 && gx < nx && gy < ny;
      }
      const int64_t g = (int64_t)gx * ny + gy;
      hv[i] = 0.0f;
      vv[i] = 0;
      zv[i] = 0;
      if (LAYERS == 2) {
        hs3[i] = 0.0f;
        sv[i] = 0;
      }
      if (ok) {
        hv[i] = snap_in[g];
        if (LAYERS == 2) hs3[i] = ssnap_in[g];
        if (row >= 1 && row <= kH3X - 2 && col >= 1 && col <= kH3Y - 2) vv[i] = v_in[g];
        if (row >= 2 && row <= kH3X - 3 && col >= 2 && col <= kH3Y - 3) {
          zv[i] = zm_in[g];
          if (LAYERS == 2) sv[i] = sm_in[g];
        }
      }
    }
    // loaded after the map loads are out, so that their wait overlaps those
    load_arrivals();
    uint16_t* s_cas = (uint16_t*)(s_casc + kH1X * kH1Y * LAYERS);  // H2 cells with a transfer: row << 8 | column
    if (threadIdx.x == 0) s_ncas = 0;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      int32_t row, col;
      if (!item(i, row, col)) continue;
      s_old[row * kH3Y + col] = hv[i];
      if (LAYERS == 2) s_sold[row * kH3Y + col] = hs3[i];
      if (row >= 1 && row <= kH3X - 2 && col >= 1 && col <= kH3Y - 2) s_vold[(row - 1) * kH2Y + col - 1] = vv[i];
      if (row >= 2 && row <= kH3X - 3 && col >= 2 && col <= kH3Y - 3) {
        s_casc[(row - 2) * kH1Y + col - 2] = zv[i];
        if (LAYERS == 2) s_sdif[(row - 2) * kH1Y + col - 2] = sv[i] - zv[i];
      }
    }
    __syncthreads();
    // start of each arrival sub-range in this tile's arrival order (read
    // after the next barrier)
    prefix_arrivals();

    // visited cells within two cells of the tile whose cascade moves
    // material: one neighbour beyond the threshold at the window's start
    // height.  The walk changes the centre only after a transfer, so a cell
    // with none such moves nothing and is skipped.  Listed in LDS so that
    // the cascades below run on full waves.
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      int32_t row, col;
      (void)item(i, row, col);
      bool act = false;
      if (vv[i] != 0) {
        const int32_t gx = x0 - 3 + row, gy = y0 - 3 + col;
        const int32_t ic = row * kH3Y + col;
        const float hc = hv[i];
        const float dd = __builtin_sqrtf(2.0f);
#pragma unroll
        for (int k = 0; k < 8; k++) {
          bool ok = true;
          if (!PERIODIC) {
            const int32_t qx = gx + c_ox[k], qy = gy + c_oy[k];
            ok = qx >= 0 && qy >= 0 && qx < nx && qy < ny;
          }
          const float diff = hc - s_old[ic + c_ox[k] * kH3Y + c_oy[k]];
          const float d = (c_ox[k] != 0 && c_oy[k] != 0) ? dd : 1.0f;
          const float excess = __builtin_fabsf(diff) - (d * ap->maxdiff) * 1.0f;
          act = act || (ok && diff != 0.0f && !(excess <= 0.0f));
        }
      }
      const uint64_t m = __ballot(act);
      const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      uint32_t base = 0;
      if ((threadIdx.x & 63) == 0 && m) base = atomicAdd(&s_ncas, (uint32_t)__popcll(m));
      base = __builtin_amdgcn_readfirstlane(base);
      if (act) s_cas[base + below] = (uint16_t)(row << 8 | col);
    }
    __syncthreads();

    // their cascades
    const uint32_t ncas = s_ncas;
    for (uint32_t i = threadIdx.x; i < ncas; i += kStepThreads) {
      const int32_t e = s_cas[i];
      const int32_t lx = (e >> 8) - 1, ly = (e & 255) - 1;  // H2 coords; H3 = +1, H1 = -1
      const uint32_t v = s_vold[lx * kH2Y + ly];
      const int32_t gx = x0 - 2 + lx, gy = y0 - 2 + ly;
      float hn[8];
      uint32_t valid = 0;
      const int32_t ic = (lx + 1) * kH3Y + (ly + 1);
#pragma unroll
      for (int k = 0; k < 8; k++) {
        hn[k] = s_old[ic + c_ox[k] * kH3Y + c_oy[k]];
        bool ok = true;
        if (!PERIODIC) {
          const int32_t qx = gx + c_ox[k], qy = gy + c_oy[k];
          ok = qx >= 0 && qy >= 0 && qx < nx && qy < ny;
        }
        valid |= (ok ? 1u : 0u) << k;
      }
      const auto sed_of = [&](int32_t k) { return s_sold[ic + off_x(k) * kH3Y + off_y(k)]; };
      int64_t centre = 0;
      cascade_cell_dev<LAYERS>(hn, sed_of, s_old[ic], LAYERS == 2 ? s_sold[ic] : 0.0f, valid,
                               settle_factor_dev(ap->settling, v), ap->maxdiff, [&](int32_t k, int64_t amt) {
                                 centre -= amt;
                                 const int32_t hx = lx - 1 + off_x(k), hy = ly - 1 + off_y(k);
                                 if (amt != 0 && hx >= 0 && hy >= 0 && hx < kH1X && hy < kH1Y)
                                   atomicAdd((unsigned long long*)&s_casc[hx * kH1Y + hy], (unsigned long long)amt);
                               });
      const int32_t hx = lx - 1, hy = ly - 1;
      if (centre != 0 && hx >= 0 && hy >= 0 && hx < kH1X && hy < kH1Y)
        atomicAdd((unsigned long long*)&s_casc[hx * kH1Y + hy], (unsigned long long)centre);
    }
    // each thread's first arrival record, loaded now so that it arrives
    // while the other threads finish their cascades and the relax ends
    if (!RELAX_ONLY) first_arrival();
    __syncthreads();

    // next snapshot for the tile and its halo.  The
    // tile's own masters seed the particle phase's pickup accumulators
    // (acc_d / acc_ds below: the front of s_work, whose relax-phase arrays
    // are dead once the cascades are summed, and clear of s_casc)
    static_assert(8 * kCell * (LAYERS == 2 ? 2 : 1) <= 4 * kH3X * kH3Y * (LAYERS == 2 ? 2 : 1) + 4 * kH2X * kH2Y,
                  "the pickup accumulators must not overlap s_casc");
    int64_t* acc_z = (int64_t*)s_work;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      int32_t row, col;
      if (!item(i, row, col) || row < 2 || row > kH3X - 3 || col < 2 || col > kH3Y - 3) continue;
      const int32_t lx = row - 2, ly = col - 2, e = lx * kH1Y + ly;  // 1-halo coordinates
      const int32_t gx = x0 - 1 + lx, gy = y0 - 1 + ly;
      const bool ok = PERIODIC || (gx >= 0 && gy >= 0 && gx < nx && gy < ny);
      const bool mine = lx >= 1 && ly >= 1 && lx <= kSX && ly <= kSY && gx < nx && gy < ny;
      const int64_t g = (int64_t)gx * ny + gy;
      const int64_t z = s_casc[e];
      const float zf = f32_from_fx(z);
      s_new[e] = ok ? zf : 0.0f;
      const int32_t li = (lx - 1) * kSY + (ly - 1);
      if (mine) {
        acc_z[li] = z;
        snap_out[g] = zf;
      }
      if (LAYERS == 2) {
        int64_t s = z + s_sdif[e];
        if (s < 0) s = 0;
        const float sf = f32_from_fx(s);
        s_snew[e] = ok ? sf : 0.0f;
        if (mine) {
          acc_z[kCell + li] = s;
          ssnap_out[g] = sf;
        }
      }
    }
    __syncthreads();
  }
  }  // relax (MODE 0, 1)
  {
    int64_t part = (int64_t)part_c + (int64_t)part_n;
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = part;
    __syncthreads();
    if (threadIdx.x == 0) {
      int64_t b0 = 0;
      for (int i = 0; i < kStepThreads / 64; i++) b0 += s_part[i];
      s_base = 9 * b0;
      s_lost = 0;
      s_far = 0;
    }
  }

  // ---------------- 2. particles of the tile ----------------
  ap = step_args(ap);
  asm volatile("" : "+s"(tp));
  int64_t* acc_d = (int64_t*)s_work;
  int64_t* acc_ds = acc_d + kCell;  // LAYERS == 2
  uint32_t* acc_v = (uint32_t*)(acc_d + kCell * (LAYERS == 2 ? 2 : 1));
  int64_t* acc_t = (int64_t*)(acc_v + kCell);  // TRACK (kCell*4), 8-byte aligned: kCell*4 bytes of acc_v
  for (int e = threadIdx.x; e < kCell; e += kStepThreads) {
    acc_v[e] = 0;  // acc_d / acc_ds hold the masters, the pickups add to them
    if (TRACK) {
      acc_t[e] = 0;
      acc_t[kCell + e] = 0;
      acc_t[2 * kCell + e] = 0;
      acc_t[3 * kCell + e] = 0;
    }
  }
  __syncthreads();  // s_rpre is read from s_slot before s_slot restarts
  if (threadIdx.x < 9) s_slot[threadIdx.x] = 0;
  __syncthreads();

  if (!RELAX_ONLY) {
    FlyConsts k;
    k.nx = nx;
    k.ny = ny;
    k.rcp_nx = rcp_nx;
    k.rcp_ny = rcp_ny;
    k.mapscale = ap->mapscale;
    k.max_age = ap->max_age;
    set_boundarylayer(k, ap->boundarylayer);
    k.suspension = ap->suspension;
    k.gravity = ap->gravity;
    k.abrasion = ap->abrasion;
    k.ps = mk(tp->ps[0], tp->ps[1], tp->ps[2]);
    k.nps = mk(tp->nps[0], tp->nps[1], tp->nps[2]);
    const uint64_t ck = cycle_key(tp->seed, cycle);
    const int64_t p0 = tp->part0;
    const int64_t out_base = s_base;  // 9 x the input counts of tiles 0 .. u-1

    // one input record
    using Rec = PRec;
    auto load = [](const PRec* in, int64_t j) __attribute__((always_inline)) { return in[j]; };
    // a particle more than one tile away goes to the far list; the tile of
    // cell (fx, fy) counts it among its next window's arrivals
    auto send_far = [&](f4a8 o0, f4a8 o1, int64_t ledger, int32_t fx, int32_t fy) __attribute__((always_inline)) {
      const int32_t dest = t0 + (fx / kSX) * tiles_y + fy / kSY;
      atomicAdd(&ap->nin_next[dest], 1u);
      atomicAdd(&ap->csum_next[dest / kChunk], 1u);
      const uint32_t fslot = atomicAdd(ap->far_cnt_out, 1u);
      ap->far_out[fslot] = PRec{o0, o1, ledger};
    };
    // step one record and write it out
    auto process = [&](const Rec& r) __attribute__((always_inline)) {
      Particle w;
      const f4a8 q0 = r.q0;
      const f4a8 q1 = r.q1;
      w.px = q0.x; w.py = q0.y; w.pz = q0.z; w.sed = q0.w;
      w.sx = q1.x; w.sy = q1.y; w.sz = q1.z;
      w.age = ap->window;
      w.ledger = r.ledger;
      w.lastc = 0;
      const uint32_t pid = f2u(q1.w);
      const uint64_t pk = particle_key(ck, (uint64_t)((int64_t)pid - p0));
      int32_t cx, cy;
      const bool ok = cell_of<PERIODIC>(w.px, w.pz, k, cx, cy);
      int64_t dead_cell = -1;
      bool dead = !ok;
      if (ok && (cx < x0 || cy < y0 || cx >= x0 + kSX || cy >= y0 + kSY)) {
        // routing always places a particle in the tile of its cell; keep
        // LDS indices in range whatever happens by forwarding a stray one
        send_far(q0, q1, w.ledger, cx, cy);
        return;
      }
      if (ok) {
        const int32_t lx = cx - x0, ly = cy - y0;
        TileMap<kH1Y> m{s_new, s_snew, (lx + 1) * kH1Y + (ly + 1)};
        TileAcc<kCell> acc{acc_d, acc_ds, acc_v, acc_t, lx * kSY + ly};
        if (fly<PERIODIC, TRACK, LAYERS>(w, pk, cx, cy, k, m, acc) == kDied) {
          dead = true;
          dead_cell = (int64_t)cx * ny + cy;
        }
      }
      if (dead) {
        // died in this call at its cell, or found off the map: the cell it left
        const int64_t c = dead_cell >= 0 ? dead_cell : (int64_t)f2u(q0.x);
        if (DEPOSIT) {
          const int32_t lx = (int32_t)(c / ny) - x0, ly = (int32_t)(c % ny) - y0;
          if (w.ledger != 0 && lx >= 0 && ly >= 0 && lx < kSX && ly < kSY) {
            const int32_t li = lx * kSY + ly;
            atomicAdd((unsigned long long*)&acc_d[li], (unsigned long long)w.ledger);
            if (LAYERS == 2) atomicAdd((unsigned long long*)&acc_ds[li], (unsigned long long)w.ledger);
          }
        } else {
          atomicAdd((unsigned long long*)&s_lost, (unsigned long long)w.ledger);
        }
        return;
      }
      // route by the cell the particle now occupies; one that leaves a
      // bounded map (or whose position stops being finite) stays with the
      // tile of its last cell and dies there at its next call
      int32_t ncx = 0, ncy = 0;
      int32_t code = 4;
      bool off = true;
      if (cell_of<PERIODIC>(w.px, w.pz, k, ncx, ncy)) {
        off = false;
        int32_t dtx = ncx / kSX - tx, dty = ncy / kSY - ty;
        if (PERIODIC) {
          if (tiles_x > 2) {
            if (dtx == tiles_x - 1) dtx = -1;
            if (dtx == 1 - tiles_x) dtx = 1;
          }
          if (tiles_y > 2) {
            if (dty == tiles_y - 1) dty = -1;
            if (dty == 1 - tiles_y) dty = 1;
          }
        }
        code = (dtx < -1 || dtx > 1 || dty < -1 || dty > 1) ? 255 : (dtx + 1) * 3 + (dty + 1);
      }
      const f4a8 o0 = off ? f4a8{u2f((uint32_t)w.lastc), w.py, __builtin_nanf(""), w.sed}
                          : f4a8{w.px, w.py, w.pz, w.sed};
      const f4a8 o1 = {w.sx, w.sy, w.sz, u2f(pid)};
      if (code == 255) {
        atomicAdd(&s_far, 1u);
        send_far(o0, o1, w.ledger, ncx, ncy);
        return;
      }
      // sub-range `code` of this tile's output region holds up to nin_u records
      const int64_t o = out_base + (int64_t)code * nin_u + atomicAdd(&s_slot[code], 1u);
      ap->out[o] = PRec{o0, o1, w.ledger};
    };

    // the arrivals, e = 0 .. n_in - 1 over the nine sub-ranges in order; each
    // thread's e increase, so its sub-range cursor only moves forward.  The
    // next record is loaded while the current one is stepped.
    const uint32_t n_in = s_rpre[9];
    uint32_t sr = sr0;
    auto index_of = [&](uint32_t e) __attribute__((always_inline)) {
      while (sr < 8 && e >= s_rpre[sr + 1]) sr++;
      return s_rbase[sr] + (int64_t)(e - s_rpre[sr]);
    };
    {
      Rec cur = rec0;
      for (uint32_t e = threadIdx.x; e < n_in; e += kStepThreads) {
        Rec nxt{};
        if (e + kStepThreads < n_in) nxt = load(ap->in, index_of(e + kStepThreads));
        process(cur);
        cur = nxt;
      }
    }
    for (int64_t j = threadIdx.x; j < (int64_t)far_n; j += kStepThreads) {
      const int64_t fp = (int64_t)f2u(ap->far_in[j].q1.w);
      if (fp < p0 || fp >= p0 + tp->npart) continue;  // another terrain's particle
      int32_t cx, cy;
      const f4a8 q0 = ap->far_in[j].q0;
      int32_t ctx, cty;
      if (cell_of<PERIODIC>(q0.x, q0.z, k, cx, cy)) {
        ctx = cx / kSX;
        cty = cy / kSY;
      } else {
        const int32_t lc = (int32_t)f2u(q0.x);
        ctx = (lc / ny) / kSX;
        cty = (lc % ny) / kSY;
      }
      if (ctx == tx && cty == ty) process(load(ap->far_in, j));
    }
  }
  __syncthreads();

  // ---------------- 3. write the tile's window results ----------------
  ap = step_args(ap);
  int64_t* zm_out = ap->zm_out + c0;
  int64_t* sm_out = LAYERS == 2 ? ap->sm_out + c0 : nullptr;
  uint32_t* v_out = ap->v_out + c0;
  int64_t* trk = TRACK ? ap->trk + c0 : nullptr;
  if (EXT) {
    snap_out = ap->snap_out + c0;
    if (LAYERS == 2) ssnap_out = ap->ssnap_out + c0;
  }
#pragma unroll
  for (int i = 0; i < kCellPer; i++) {
    const int e = threadIdx.x + i * kStepThreads;
    const int32_t gx = x0 + e / kSY, gy = y0 + e % kSY;
    if (e >= kCell || gx >= nx || gy >= ny) continue;
    const int64_t g = (int64_t)gx * ny + gy;
    // master with this window's pickups; the clamp of the sediment layer at
    // zero follows the next window's cascades
    zm_out[g] = acc_d[e];
    v_out[g] = acc_v[e];
    if (LAYERS == 2) sm_out[g] = acc_ds[e];
    if (EXT) {  // the snapshot the colour-ordered relax starts from
      snap_out[g] = f32_from_fx(acc_d[e]);
      if (LAYERS == 2) ssnap_out[g] = f32_from_fx(acc_ds[e]);
    }
  }
  // flow tracks of the cells this window's particles visited, read here
  // rather than prefetched (16 fewer vector registers through the particle
  // loop lets five workgroups share a CU): the loads are issued now and the
  // sums stored at the very end, after the rest of the write-out
  int64_t tv[TRACK && !RELAX_ONLY ? kCellPer : 1][4], old[TRACK && !RELAX_ONLY ? kCellPer : 1][4];
  int64_t gi[TRACK && !RELAX_ONLY ? kCellPer : 1];
  if (TRACK && !RELAX_ONLY) {
#pragma unroll
    for (int i = 0; i < kCellPer; i++) {
      const int e = threadIdx.x + i * kStepThreads;
      const int32_t gx = x0 + e / kSY, gy = y0 + e % kSY;
      const bool in = e < kCell && gx < nx && gy < ny;
      gi[i] = (int64_t)gx * ny + gy;
#pragma unroll
      for (int f = 0; f < 4; f++) tv[i][f] = in ? acc_t[f * kCell + (in ? e : 0)] : 0;
    }
#pragma unroll
    for (int i = 0; i < kCellPer; i++)
#pragma unroll
      for (int f = 0; f < 4; f++) old[i][f] = tv[i][f] != 0 ? trk[f * ap->ncell + gi[i]] : 0;
  }
  // s_rbase is free again (the arrivals are consumed): it carries the chunk
  // of each direction's destination tile to the aggregation below
  int32_t* s_dchunk = (int32_t*)s_rbase;
  if (threadIdx.x < 9) {
    // particles sent towards direction d: sub-range d of this tile's output,
    // and the next window's arrivals of the tile in direction d
    const int32_t d = threadIdx.x;
    const uint32_t n = s_slot[d];
    ap->sub_base_cur[(int64_t)u * 9 + d] = s_base + (int64_t)d * nin_u;
    ap->sub_cnt_cur[(int64_t)u * 9 + d] = n;
    int32_t chunk = -1;
    if (n) {
      const int32_t dx = d / 3 - 1, dy = d % 3 - 1;
      int32_t dtx = tx + dx, dty = ty + dy;
      if (PERIODIC) {
        dtx = wrapt(dtx, tiles_x);
        dty = wrapt(dty, tiles_y);
      }
      const int32_t dest = t0 + dtx * tiles_y + dty;
      atomicAdd(&ap->nin_next[dest], n);
      chunk = dest / kChunk;
    }
    s_dchunk[d] = chunk;
  }
  if (threadIdx.x == 0) {
    ap->nin_clear[u] = 0;  // the window after next accumulates here
    if (u % kChunk == 0) ap->csum_clear[u / kChunk] = 0;
    if (u == 0) {
      *ap->far_cnt_clear = 0;
      if ((hs | ls) > 0)
        for (int i = 0; i < 16; i++) ap->hcnt_clear[i] = 0;
    }
    // crowded (or light) now: listed for the next launch (the count moves
    // little from one window to the next)
    if (hs > 0 && nin_u > kHeavyMin) {
      const uint32_t home = home_of((uint32_t)u);
      const uint32_t slot = atomicAdd(&ap->hcnt_next[home], 1u);
      if (slot < hs / 8) {
        ap->heavy_next[home * (hs / 8) + slot] = (uint32_t)u;
        ap->hstamp[u] = (uint32_t)ap->window + 2u;
      }
    } else if (ls > 0 && nin_u <= kLightMax) {
      const uint32_t home = home_of((uint32_t)u);
      const uint32_t slot = atomicAdd(&ap->hcnt_next[8 + home], 1u);
      if (slot < ls / 8) {
        ap->heavy_next[kHeavySlotsMax + home * (ls / 8) + slot] = (uint32_t)u;
        ap->hstamp[u] = (uint32_t)ap->window + 2u;
      }
    }
  }
  __syncthreads();
  if (!RELAX_ONLY && threadIdx.x < 9) {
    // chunk sums of the next window's arrivals: one atomic per distinct chunk
    // (the nine destinations mostly share one or two), by the thread of the
    // chunk's first direction
    const int d = threadIdx.x;
    const int32_t ch = s_dchunk[d];
    bool first = ch >= 0;
#pragma unroll
    for (int e = 0; e < 9; e++) first = first && !(e < d && s_dchunk[e] == ch);
    if (first) {
      uint32_t n = 0;
#pragma unroll
      for (int e = 0; e < 9; e++) n += e >= d && s_dchunk[e] == ch ? s_slot[e] : 0u;
      atomicAdd(&ap->csum_next[ch], n);
    }
  }
  if (!RELAX_ONLY && threadIdx.x == 0) {
    // statistics: one atomic per workgroup and kind; a particle that made its
    // step was sent on, to a sub-range or the far list
    const uint64_t far = s_far;
    uint64_t steps = far;
    for (int d = 0; d < 9; d++) steps += s_slot[d];
    const uint32_t slot = (uint32_t)u & (kStatSlots - 1);
    if (steps) atomicAdd((unsigned long long*)&ap->stat[kStatSteps * kStatSlots + slot], (unsigned long long)steps);
    if (far) atomicAdd((unsigned long long*)&ap->stat[kStatFar * kStatSlots + slot], (unsigned long long)far);
    if (nin_u) atomicMax((unsigned long long*)&ap->stat[kStatMaxTile * kStatSlots + slot], (unsigned long long)nin_u);
    if (nin_u > kCrowded) atomicAdd((unsigned long long*)&ap->stat[kStatCrowded * kStatSlots + slot], 1ull);
    if (listed) {
      const bool light_slot = blockIdx.x >= (uint32_t)(ap->heavy_slots + ap->default_slots);
      atomicAdd((unsigned long long*)&ap->stat[(light_slot ? kStatLight : kStatHeavy) * kStatSlots + slot], 1ull);
    }
  }
  if (!DEPOSIT && threadIdx.x == 0) {
    const int64_t l = s_lost;
    if (l != 0)
      atomicAdd((unsigned long long*)&ap->lost[(int64_t)ap->tile_terrain[u] * kLostSlots + (u & (kLostSlots - 1))],
                (unsigned long long)l);
  }
  if (TRACK && !RELAX_ONLY) {
#pragma unroll
    for (int i = 0; i < kCellPer; i++)
#pragma unroll
      for (int f = 0; f < 4; f++)
        if (tv[i][f] != 0) trk[f * ap->ncell + gi[i]] = old[i][f] + tv[i][f];
  }
}

// Bound by the latency of a workgroup's phases (halo load, cascades,
// particles, write-out) and by vector issue within them.  Phase-wise argument
// reads, one address per halo cell and branch-free primitives took the
// kernel from 10,470 to 7,000 instructions (70 to 46 KB of code, past and
// within the instruction cache); with the lists of a one-round launch dropped
// and the cascade walk's chain shortened a window takes 14.6 us (18.8 before)
// on 256^2 with 2,000 particles, 13.2 (17.2) on 75 x 101 with 300, and 71
// (73) on 1024^2 with a million, where vector issue is half the time.
template <int SX, int SY, int NT, int WPE, bool PERIODIC, bool TRACK, int LAYERS, bool DEPOSIT, int MODE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE))) void k_step(StepArgs) {
  step_body<SX, SY, NT, PERIODIC, TRACK, LAYERS, DEPOSIT, MODE>();  // reads its arguments from the kernel argument segment
}

// The colour-ordered cascade in the same single launch per window: the tile
// re-runs, on an LDS copy of the masters, the cascades of all visited cells
// within the reach of its own cells and their one-cell halo (colour_halo: a
// bound, not a search of what they depend on), instead of one launch per
// class over the map (9 to 25 launches, each two memory round trips: 7.5 us
// apiece on 512^2).  colour_fused has the line between the two.
// Redundant work is 3.4 regions per tile, but a window pays one launch and
// one load of the region; its time is the most crowded tile's rounds of
// dependent cascades (1,500 to 5,000 cycles each).  Measured against the
// class launches: 512^2 bounded, 4096 particles 46.1 -> 12.8 ms a cycle; 400 x
// 301 periodic, two layers, 30,000 particles 85.3 -> 28.2 ms; 1024^2 with a
// million particles, where a class launch fills the chip, 110 -> 92 ms.
template <int SX, int SY, int NT, bool PERIODIC, bool TRACK, int LAYERS, bool DEPOSIT, int MODE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_colour_step(StepArgs) {
  step_body<SX, SY, NT, PERIODIC, TRACK, LAYERS, DEPOSIT, MODE>();  // reads its arguments from the kernel argument segment
}

// ---------------------------------------------------------------------------
// Launchers of one shape (instantiated per shape in swe_step_shapes.hip)
// ---------------------------------------------------------------------------
template <int SX, int SY, int NT, int WPE>
struct StepLauncher {
  template <bool P, bool T, int L, bool D>
  static void step4(const StepArgs& a, int mode, hipStream_t s) {
    const unsigned g = (unsigned)(a.heavy_slots + a.default_slots + a.light_slots);
    if (mode >= 3) {
      ColourHalo h = kColourHalo;  // the larger of the launch's two regions
      h.xl = a.chalo.xl > h.xl ? a.chalo.xl : h.xl;
      h.xh = a.chalo.xh > h.xh ? a.chalo.xh : h.xh;
      h.yl = a.chalo.yl > h.yl ? a.chalo.yl : h.yl;
      h.yh = a.chalo.yh > h.yh ? a.chalo.yh : h.yh;
      const unsigned lds = (unsigned)colour_lds(StepShape{SX, SY, NT, WPE}, h, T, L);
      if (mode == 3)
        hipLaunchKernelGGL((k_colour_step<SX, SY, NT, P, T, L, D, 3>), dim3(g), dim3(NT), lds, s, a);
      else
        hipLaunchKernelGGL((k_colour_step<SX, SY, NT, P, T, L, D, 4>), dim3(g), dim3(NT), lds, s, a);
    } else if (mode == 1)
      hipLaunchKernelGGL((k_step<SX, SY, NT, WPE, P, T, L, D, 1>), dim3(g), dim3(NT), 0, s, a);
    else if (mode == 2)
      hipLaunchKernelGGL((k_step<SX, SY, NT, WPE, P, T, L, D, 2>), dim3(g), dim3(NT), 0, s, a);
    else
      hipLaunchKernelGGL((k_step<SX, SY, NT, WPE, P, T, L, D, 0>), dim3(g), dim3(NT), 0, s, a);
  }
  template <bool P, bool T, int L>
  static void step3(const StepArgs& a, int ro, bool dep, hipStream_t s) {
    if (dep) step4<P, T, L, true>(a, ro, s);
    else step4<P, T, L, false>(a, ro, s);
  }
  template <bool P, bool T>
  static void step2(const StepArgs& a, int ro, bool dep, int layers, hipStream_t s) {
    if (layers == 2) step3<P, T, 2>(a, ro, dep, s);
    else step3<P, T, 1>(a, ro, dep, s);
  }
  template <bool P>
  static void step1(const StepArgs& a, int ro, bool dep, bool trk, int layers, hipStream_t s) {
    if (trk) step2<P, true>(a, ro, dep, layers, s);
    else step2<P, false>(a, ro, dep, layers, s);
  }
  static void launch(const StepArgs& a, bool periodic, bool track, int layers, bool deposit, int mode,
                     hipStream_t s) {
    if (periodic) step1<true>(a, mode, deposit, track, layers, s);
    else step1<false>(a, mode, deposit, track, layers, s);
  }
};

}  // namespace swe
