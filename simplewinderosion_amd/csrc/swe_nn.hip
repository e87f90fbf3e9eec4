// swe_nn.hip -- kernels of the learned surrogate (a periodic convolutional
// encoder-decoder that predicts K map-cycles of erosion at once): 3x3
// convolutions on BF16 MFMA (v_mfma_f32_16x16x32_bf16, FP32 accumulation)
// forward, data gradient (the forward kernel on flipped weights) and weight
// gradient, plus the elementwise, pooling, loss, optimiser and fixed-point
// mass-projection kernels around them.
//
// Activations are NHWC (channels contiguous), bf16; weights [Cout][9][Cin]
// bf16 with tap t = 3*(dy+1) + (dx+1); padding is periodic, like the maps.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/swe_nn.h"

static_assert(sizeof(swe_nn_adam_seg) == 72, "swe_nn_adam_seg: six pointers, two int64, two int32");

namespace swenn {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(bf16 v) { return (float)v; }
__device__ __forceinline__ bf16 f2bf(float v) { return (bf16)v; }  // round to nearest even

__device__ __forceinline__ int32_t wrapi(int32_t v, int32_t n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

// Epilogue of the tile kernels: bias, ACT (0 none, 1 ReLU, 2 zero where mask
// <= 0) and the stores of a wave's PF x CF result fragments for the tile at
// (y0, x0) of image n.
template <int PF, int CF, int S, int ACT>
__device__ __forceinline__ void conv_store(const f32x4 (&acc)[PF][CF], const float* s_bias,
                                           const bf16* __restrict__ mask, bf16* __restrict__ y16,
                                           float* __restrict__ y32, int32_t n, int32_t y0, int32_t x0, int32_t H,
                                           int32_t W, int32_t Cout, int32_t co0, int32_t vec) {
  constexpr int CP = CF == 1 ? 1 : CF / 2;  // output vectors a lane holds per pixel
  constexpr int CV = CF == 1 ? 4 : 8;       // channels of one
  const int32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rl = lane & 15, g = lane >> 4;
  // output positions of this lane: pixel rl of each fragment
  int32_t po[PF];
#pragma unroll
  for (int f = 0; f < PF; f++) {
    const int32_t idx = wave * PF + f, yy = y0 + idx / S, xx = x0 + 16 * (idx % S) + rl;
    po[f] = yy < H && xx < W ? (n * H + yy) * W + xx : -1;
  }
  typedef bf16 bf16v __attribute__((ext_vector_type(CV)));
  bf16v mk[ACT == 2 ? PF : 1][ACT == 2 ? CP : 1];
  if (ACT == 2 && vec) {  // every mask load in flight at once
#pragma unroll
    for (int f = 0; f < PF; f++)
#pragma unroll
      for (int q = 0; q < CP; q++) {
        const int32_t co = co0 + 32 * q + CV * g;
        if (po[f] >= 0 && co < Cout) mk[f][q] = *(const bf16v*)(mask + (int64_t)po[f] * Cout + co);
      }
  }
#pragma unroll
  for (int f = 0; f < PF; f++) {
    if (po[f] < 0) continue;
#pragma unroll
    for (int q = 0; q < CP; q++) {
      const int32_t co = co0 + 32 * q + CV * g;
      if (co >= Cout) continue;
      float v[CV];
#pragma unroll
      for (int e = 0; e < CV; e++) {
        v[e] = acc[f][CF == 1 ? 0 : 2 * q + e / 4][e % 4] + s_bias[32 * q + CV * g + e];
        if (ACT == 1) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
      }
      const int64_t o = (int64_t)po[f] * Cout + co;
      if (vec) {
        // all CV channels lie below Cout and the vectors are aligned
        if (ACT == 2) {
#pragma unroll
          for (int e = 0; e < CV; e++) v[e] = bf2f(mk[f][q][e]) > 0.0f ? v[e] : 0.0f;
        }
        if (y16) {
          bf16v r;
#pragma unroll
          for (int e = 0; e < CV; e++) r[e] = f2bf(v[e]);
          *(bf16v*)(y16 + o) = r;
        }
        if (y32) {
#pragma unroll
          for (int e = 0; e < CV; e += 4) *(f32x4*)(y32 + o + e) = (f32x4){v[e], v[e + 1], v[e + 2], v[e + 3]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < CV; e++) {
          if (co + e >= Cout) continue;
          if (ACT == 2) v[e] = bf2f(mask[o + e]) > 0.0f ? v[e] : 0.0f;
          if (y16) y16[o + e] = f2bf(v[e]);
          if (y32) y32[o + e] = v[e];
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// 3x3 convolution over rectangular tiles: a workgroup (4 waves) owns 64 PF
// pixels (4 PF / S rows of 16 S columns of one image) x 16 CF output
// channels.  This kernel takes up to 32 input channels: the weights of all
// nine taps are staged in LDS once, then for each of the workgroup's `per`
// consecutive tiles the input patch (the tile and its one-pixel periodic
// halo, read once for all nine taps); the next tile's loads are in flight
// while the waves compute.
// LDS rows are one pixel (one output channel of one tap) of 32 channels, 64
// bytes at a stride of 80, so that the 16 rows a fragment read touches fall
// in different banks and a tap is an immediate offset.
//
// The weights are the MFMA's A operand and the pixels its B operand, so a
// lane's four results are four output channels of one pixel.  Two fragments
// interleave their rows (row r of fragment j is channel 8 (r / 4) + 4 j +
// r % 4 of their 32), which leaves a lane with eight consecutive channels:
// one 16-byte store (and mask load) where a pixel-major result takes eight
// two-byte ones.  Each wave takes PF fragments of 16 pixels and all CF of
// channels: PF + CF reads of 1 KB for PF CF MFMAs.
//
// Tiles are dealt so that each XCD (workgroup b runs on XCD b % 8) gets a
// contiguous range with all its channel blocks.
//
// Bound: memory at full resolution (32 -> 32 moves 67 MB, 100 with a mask).
// Against a row-streamed kernel with pixel-major results (us, batch 8): 32 ->
// 32 at 256^2 25.3 -> 20.6, its masked data gradient 31.0 -> 24.3; 8 -> 32
// 25.2 -> 19.9; 32 -> 16 20.6 -> 13.5; 32 -> 32 at 200 x 230, batch 3, 13.0 ->
// 10.1.
// ---------------------------------------------------------------------------
// waves per SIMD that the LDS of a shape leaves room for, and its register budget
// (the 16-channel shape fits four waves' registers but for two)
constexpr int conv_tile_waves(int pf, int cf) { return cf == 4 ? 2 : (pf == 4 && cf == 2 ? 3 : 4); }
constexpr int conv_tile_budget(int pf, int cf) { return cf == 1 ? 3 : conv_tile_waves(pf, cf); }

template <int PF, int CF, int S, int ACT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(conv_tile_budget(PF, CF)))) void k_conv_tile(
    const bf16* __restrict__ x, const bf16* __restrict__ w, const float* __restrict__ bias,
    const bf16* __restrict__ mask, bf16* __restrict__ y16, float* __restrict__ y32, int32_t N, int32_t H, int32_t W,
    int32_t Cin, int32_t Cout, int32_t per, int32_t vec) {
  constexpr int TW = 16 * S, TH = 4 * PF / S;  // tile columns, rows
  constexpr int PW = TW + 2, PH = TH + 2;      // patch
  constexpr int LD = 40;                       // LDS row stride (elements)
  constexpr int AI = PW * PH * 4, AP = (AI + 255) / 256;    // 16-byte items of the patch, per thread
  constexpr int BR = 9 * 16 * CF, BP = (BR * 4 + 255) / 256;  // weight rows; items per thread
  __shared__ __attribute__((aligned(16))) bf16 s_a[PW * PH * LD];
  __shared__ __attribute__((aligned(16))) bf16 s_b[BR * LD];
  __shared__ __attribute__((aligned(16))) float s_bias[16 * CF];
  const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t rl = lane & 15, g = lane >> 4, gg = tid & 3;
  const int32_t tx = (W + TW - 1) / TW, ty = (H + TH - 1) / TH, tiles = N * ty * tx;
  const int32_t ncob = (Cout + 16 * CF - 1) / (16 * CF);
  const int32_t groups = (tiles + per - 1) / per;
  // this workgroup's (tile group, channel block): XCD k takes the groups from
  // k q + min(k, r) on
  const uint32_t nb = gridDim.x, b = blockIdx.x, q8 = nb / 8, r8 = nb % 8, xcd = b % 8;
  const int32_t lin = (int32_t)(xcd * q8 + (xcd < r8 ? xcd : r8) + b / 8);
  const int32_t grp = lin / ncob, co0 = (lin - grp * ncob) * 16 * CF;
  if (grp >= groups) return;
  const int32_t t_first = grp * per, t_end = t_first + per < tiles ? t_first + per : tiles;

  constexpr uint32_t kBad = 0x80000000u;  // past both buffers: reads zero
  constexpr int kRawFlags = 0x00020000;
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, (int)((int64_t)N * H * W * Cin * 2), kRawFlags);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, (int)((int64_t)Cout * 9 * Cin * 2), kRawFlags);
  // weight items: LDS row (tap, fragment, row) <- the channel it stands for
  bf16x8 rb[BP];
#pragma unroll
  for (int h = 0; h < BP; h++) {
    const int32_t rho = (tid + 256 * h) >> 2, t = rho / (16 * CF), jr = rho % (16 * CF), j = jr >> 4, r = jr & 15;
    const int32_t co = co0 + (CF == 1 ? r : 32 * (j >> 1) + 8 * (r >> 2) + 4 * (j & 1) + (r & 3));
    const uint32_t o = rho < BR && co < Cout && 8 * gg < Cin ? (uint32_t)(((co * 9 + t) * Cin + 8 * gg) * 2) : kBad;
    rb[h] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, (int)o, 0, 0));
  }
  uint32_t io[AP];  // byte offsets of the patch items of the tile being loaded
  // on maps of at least a patch a row or column wraps at most once: an
  // item's offset in the patch is fixed and its wraps are two compares
  const bool big = H >= PH && W >= PW;
  const uint32_t rowb = (uint32_t)(W * Cin * 2), imgb = (uint32_t)H * rowb;
  auto place = [&](int32_t tile) __attribute__((always_inline)) {
    // (the items' rows and columns are recomputed each time: held over the
    // tiles they would take 30 registers)
    int32_t it = tid;
    asm volatile("" : "+v"(it));
    const int32_t cx = tile % tx, cy = (tile / tx) % ty, n = tile / (tx * ty);
    // (H and W may be smaller than a patch)
    const int32_t by = (cy * TH + H - 1) % H, bx = (cx * TW + W - 1) % W;
    if (big) {
      const uint32_t base = (uint32_t)n * imgb + (uint32_t)by * rowb + (uint32_t)(bx * Cin * 2);
#pragma unroll
      for (int h = 0; h < AP; h++) {
        const int32_t p = (it + 256 * h) >> 2, r = p / PW, c = p - r * PW;
        uint32_t o = base + (uint32_t)r * rowb + (uint32_t)(c * Cin * 2 + 16 * gg);
        if (r >= H - by) o -= imgb;
        if (c >= W - bx) o -= rowb;
        io[h] = p < PW * PH ? o : kBad;
      }
      return;
    }
#pragma unroll
    for (int h = 0; h < AP; h++) {
      const int32_t p = (it + 256 * h) >> 2, r = p / PW, c = p - r * PW;
      int32_t yy = by + r, xx = bx + c;
      if (yy >= H) yy = yy < 2 * H ? yy - H : yy % H;
      if (xx >= W) xx = xx < 2 * W ? xx - W : xx % W;
      io[h] = p < PW * PH ? (uint32_t)((((n * H + yy) * W + xx) * Cin + 8 * gg) * 2) : kBad;
    }
  };
  bf16x8 ra[AP];
  const bool gok = 8 * gg < Cin;
  auto load_a = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < AP; h++)
      ra[h] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(gok ? io[h] : kBad), 0, 0));
  };
  auto store_a = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < AP; h++) {
      const int32_t p = (tid + 256 * h) >> 2;
      if (AI % 256 == 0 || p < PW * PH) *(bf16x8*)&s_a[p * LD + 8 * gg] = ra[h];
    }
  };
  if (tid < 16 * CF) s_bias[tid] = bias && co0 + tid < Cout ? bias[co0 + tid] : 0.0f;

  place(t_first);
  load_a();
#pragma unroll
  for (int h = 0; h < BP; h++) {
    const int32_t rho = (tid + 256 * h) >> 2;
    if (BR * 4 % 256 == 0 || rho < BR) *(bf16x8*)&s_b[rho * LD + 8 * gg] = rb[h];
  }
  store_a();
  __syncthreads();
  // fragment addresses: pixel (row, segment) of fragment f of this wave
  const bf16* ap[PF];
#pragma unroll
  for (int f = 0; f < PF; f++) {
    const int32_t idx = wave * PF + f;
    ap[f] = s_a + ((idx / S) * PW + 16 * (idx % S) + rl) * LD + 8 * g;
  }
  const bf16* bp = s_b + rl * LD + 8 * g;

  for (int32_t tile = t_first; tile < t_end; tile++) {
    f32x4 acc[PF][CF];
#pragma unroll
    for (int f = 0; f < PF; f++)
#pragma unroll
      for (int j = 0; j < CF; j++) acc[f][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    const bool more = tile + 1 < t_end;
    if (more) {
      place(tile + 1);
      load_a();
    }
    // a row of taps at a time: unrolled over all nine, the scheduler reads
    // fragments so far ahead that they spill
#pragma unroll 1
    for (int dy = 0; dy < 3; dy++) {
      const bf16* bt = bp + dy * 3 * CF * 16 * LD;
      const int32_t at = dy * PW * LD;
#pragma unroll
      for (int dx = 0; dx < 3; dx++) {
        bf16x8 fa[CF], fb[PF];
#pragma unroll
        for (int j = 0; j < CF; j++) fa[j] = *(const bf16x8*)(bt + (dx * CF + j) * 16 * LD);
#pragma unroll
        for (int f = 0; f < PF; f++) fb[f] = *(const bf16x8*)(ap[f] + at + dx * LD);
#pragma unroll
        for (int f = 0; f < PF; f++)
#pragma unroll
          for (int j = 0; j < CF; j++)
            acc[f][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[j], fb[f], acc[f][j], 0, 0, 0);
      }
    }
    if (more) {
      __syncthreads();
      store_a();
      __syncthreads();
    }
    conv_store<PF, CF, S, ACT>(acc, s_bias, mask, y16, y32, tile / (tx * ty), (tile / tx) % ty * TH, tile % tx * TW, H, W,
                               Cout, co0, vec);
  }
}

// ---------------------------------------------------------------------------
// The same convolution for more than 32 input channels.  The tile's whole
// patch (up to KC = 256 channels; more run as blocks of KC) stays in LDS, and
// the weights stream through it tap by tap, two taps ahead in registers: so
// the reduction runs tap by tap and within a tap over the 32-channel chunks,
// the order of the implicit GEMM's k = tap Cin + channel; with several blocks of
// KC, block by block.  With kz > 1 the k-steps are summed in kz slices
// [z K / kz, (z + 1) K / kz) whose sums are added in order (a layer given the
// workspace of a split reduction).
// LDS rows are KC channels at a stride of KC + 8 elements (16 m + 4 dwords:
// the 16 rows of a fragment read fall in different banks).
//
// Bound: LDS reads and the barrier a tap (PF + CF reads of 1 KB feed PF CF
// MFMAs, two chunks' reads ahead of them; 38% of the MFMA rate a large product
// reaches at 128 -> 128).  Against a flattened-pixel kernel that staged every
// tap's pixels anew, with the split reduction's partial sums through memory
// (us, batch 8, forward / masked data gradient): 64 -> 64 at 128^2 28.4 / 33.5
// -> 20.4 / 23.7; 128 -> 128 at 64^2 27.6 / 32.2 -> 18.3 / 18.9; 192 -> 192 at
// 32^2 28.4 / 28.0 -> 17.8 / 18.5; 256 -> 192 at 16^2 18.6 / 17.1 -> 14.0 /
// 11.9; 64 -> 64 at 512^2, batch 1, 50.9 / 63.9 -> 40.3 / 42.9.  Reading one
// chunk ahead across the taps' barriers took 10% longer (spills at 4 x 4), four
// chunks at once 10% longer in the smallest shapes; the weights' loads a tap
// earlier 7% longer at 4 x 4.
// ---------------------------------------------------------------------------
// 32-channel chunks of a block at most: KC <= 256, for the largest workgroups
// 192 (their patch of more would not fit the LDS).  Those hold two workgroups a
// CU at 256 registers, of which about 20 spill (80 to 88 bytes of scratch).
constexpr int conv_wide_chunks(int pf, int cf) { return pf * cf > 8 ? 6 : 8; }

template <int PF, int CF, int S, int ACT, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SPLIT && PF * CF > 4 ? 1 : 2))) void k_conv_wide(
    const bf16* __restrict__ x, const bf16* __restrict__ w, const float* __restrict__ bias,
    const bf16* __restrict__ mask, bf16* __restrict__ y16, float* __restrict__ y32, int32_t N, int32_t H, int32_t W,
    int32_t Cin, int32_t Cout, int32_t KC, int32_t kz, int32_t two, int32_t vec) {
  constexpr int TW = 16 * S, TH = 4 * PF / S, PW = TW + 2, PH = TH + 2, NP = PW * PH;
  constexpr int AP = (NP + 63) / 64;                // patch pixels per thread quad
  constexpr int RB = 16 * CF;                       // weight rows of a tap
  constexpr int QB = 64 / RB;                       // chunks the 64 quads load at once
  constexpr int BP = (conv_wide_chunks(PF, CF) + QB - 1) / QB;  // weight loads a thread holds of one tap
  extern __shared__ __attribute__((aligned(16))) bf16 s_wide[];
  const int32_t LD = KC + 8, nc = KC / 32;
  bf16* s_a = s_wide;
  bf16* s_b = s_wide + NP * LD;
  float* s_bias = (float*)(s_b + (two ? 2 : 1) * RB * LD);
  const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t rl = lane & 15, g = lane >> 4, gg = tid & 3, quad = tid >> 2;
  const int32_t tx = (W + TW - 1) / TW, ty = (H + TH - 1) / TH;
  const int32_t ncob = (Cout + RB - 1) / RB;
  const uint32_t nb = gridDim.x, b = blockIdx.x, q8 = nb / 8, r8 = nb % 8, xcd = b % 8;
  const int32_t lin = (int32_t)(xcd * q8 + (xcd < r8 ? xcd : r8) + b / 8);
  const int32_t tile = lin / ncob, co0 = (lin - tile * ncob) * RB;
  const int32_t cx = tile % tx, cy = (tile / tx) % ty, n = tile / (tx * ty);

  constexpr uint32_t kBad = 0x80000000u;
  constexpr int kRawFlags = 0x00020000;
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, (int)((int64_t)N * H * W * Cin * 2), kRawFlags);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, (int)((int64_t)Cout * 9 * Cin * 2), kRawFlags);
  uint32_t io[AP];
  {
    const int32_t by = (cy * TH + H - 1) % H, bx = (cx * TW + W - 1) % W;
#pragma unroll
    for (int h = 0; h < AP; h++) {
      const int32_t p = quad + 64 * h, r = p / PW, c = p - r * PW;
      int32_t yy = by + r, xx = bx + c;
      if (yy >= H) yy = yy < 2 * H ? yy - H : yy % H;
      if (xx >= W) xx = xx < 2 * W ? xx - W : xx % W;
      io[h] = p < NP ? (uint32_t)((((n * H + yy) * W + xx) * Cin + 8 * gg) * 2) : kBad;
    }
  }
  // weights: quad -> (row of the tap's block, chunk within a group of QB)
  const int32_t brow = quad % RB, bq = quad / RB;
  uint32_t wo;
  {
    const int32_t j = brow >> 4, r = brow & 15;
    const int32_t co = co0 + (CF == 1 ? r : 32 * (j >> 1) + 8 * (r >> 2) + 4 * (j & 1) + (r & 3));
    wo = co < Cout ? (uint32_t)((co * 9 * Cin + 8 * gg) * 2) : kBad;
  }
  // the weights of tap t of channel block k0 (zero past Cin and Cout)
  struct Tap {
    bf16x8 v[BP];
  };
  auto load_b = [&](Tap& r, int32_t t, int32_t k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BP; i++) {
      if (QB * i >= nc) continue;
      const int32_t k = k0 + 32 * (QB * i + bq);
      const bool ok = wo != kBad && k + 8 * gg < Cin;
      r.v[i] = __builtin_bit_cast(
          bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, (int)(ok ? wo + (uint32_t)((t * Cin + k) * 2) : kBad), 0, 0));
    }
  };
  auto store_b = [&](const Tap& r, int32_t buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BP; i++) {
      if (QB * i >= nc) continue;
      const int32_t c = QB * i + bq;
      if (c < nc) *(bf16x8*)&s_b[(buf * RB + brow) * LD + 32 * c + 8 * gg] = r.v[i];
    }
  };
  if (tid < RB) s_bias[tid] = bias && co0 + tid < Cout ? bias[co0 + tid] : 0.0f;

  const bf16* ap[PF];
#pragma unroll
  for (int f = 0; f < PF; f++) {
    const int32_t idx = wave * PF + f;
    ap[f] = s_a + ((idx / S) * PW + 16 * (idx % S) + rl) * LD + 8 * g;
  }
  const bf16* bp = s_b + rl * LD + 8 * g;
  f32x4 acc[PF][CF], tot[SPLIT ? PF : 1][SPLIT ? CF : 1];
#pragma unroll
  for (int f = 0; f < PF; f++)
#pragma unroll
    for (int j = 0; j < CF; j++) acc[f][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  // split reduction: the slice that ends before step `cut`
  const int32_t ksteps = 9 * ((Cin + 31) / 32);
  int32_t z = 0, step = 0, cut = SPLIT && kz > 1 ? ksteps / kz : ksteps;
  auto slice_end = [&]() __attribute__((always_inline)) {
    if (SPLIT && step == cut && step < ksteps) {
#pragma unroll
      for (int f = 0; f < PF; f++)
#pragma unroll
        for (int j = 0; j < CF; j++) {
          tot[f][j] = z == 0 ? acc[f][j] : tot[f][j] + acc[f][j];
          acc[f][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        }
      z++;
      cut = (int32_t)((int64_t)(z + 1) * ksteps / kz);
    }
  };

  for (int32_t k0 = 0; k0 < Cin; k0 += KC) {
    Tap w0, w1;
    load_b(w0, 0, k0);
    // the patch, two or four chunks of loads in flight at a time
    constexpr int AB = PF == 4 ? 2 : 4;
    if (k0 > 0) __syncthreads();  // the previous block's reads are done
    for (int32_t c0 = 0; c0 < nc; c0 += AB) {
      bf16x8 ra[AB][AP];
#pragma unroll
      for (int c = 0; c < AB; c++) {
        const bool ok = c0 + c < nc && k0 + 32 * (c0 + c) + 8 * gg < Cin;
#pragma unroll
        for (int h = 0; h < AP; h++)
          ra[c][h] = __builtin_bit_cast(
              bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                          xr, (int)(ok && io[h] != kBad ? io[h] + (uint32_t)(2 * k0 + 64 * (c0 + c)) : kBad), 0, 0));
      }
#pragma unroll
      for (int c = 0; c < AB; c++) {
        if (c0 + c >= nc) continue;
#pragma unroll
        for (int h = 0; h < AP; h++) {
          const int32_t p = quad + 64 * h;
          if (NP % 64 == 0 || p < NP) *(bf16x8*)&s_a[p * LD + 32 * (c0 + c) + 8 * gg] = ra[c][h];
        }
      }
    }
    store_b(w0, 0);
    load_b(w1, 1, k0);
    __syncthreads();
    // chunks of this block that hold channels (the steps of the GEMM)
    const int32_t ncb = (Cin - k0 + 31) / 32 < nc ? (Cin - k0 + 31) / 32 : nc;
#pragma unroll
    for (int t = 0; t < 9; t++) {
      // with two weight buffers the next tap's go to the other one here
      if (two && t + 1 < 9) store_b(t % 2 == 0 ? w1 : w0, (t + 1) & 1);
      if (t + 2 < 9) load_b(t % 2 == 0 ? w0 : w1, t + 2, k0);
      const bf16* bt = bp + (two ? (t & 1) * RB * LD : 0);
      const int32_t at = ((t / 3) * PW + t % 3) * LD;
      for (int32_t c = 0; c < ncb; c += 2) {
        bf16x8 fa[2][CF], fb[2][PF];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          if (u == 1 && c + 1 >= ncb) continue;
#pragma unroll
          for (int j = 0; j < CF; j++) fa[u][j] = *(const bf16x8*)(bt + j * 16 * LD + 32 * (c + u));
#pragma unroll
          for (int f = 0; f < PF; f++) fb[u][f] = *(const bf16x8*)(ap[f] + at + 32 * (c + u));
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
          if (u == 1 && c + 1 >= ncb) continue;
#pragma unroll
          for (int f = 0; f < PF; f++)
#pragma unroll
            for (int j = 0; j < CF; j++)
              acc[f][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[u][j], fb[u][f], acc[f][j], 0, 0, 0);
          step++;
          slice_end();
        }
      }
      if (t + 1 < 9) {
        __syncthreads();
        if (!two) {
          store_b(t % 2 == 0 ? w1 : w0, 0);
          __syncthreads();
        }
      }
    }
  }
  if (SPLIT && z > 0) {
#pragma unroll
    for (int f = 0; f < PF; f++)
#pragma unroll
      for (int j = 0; j < CF; j++) acc[f][j] = tot[f][j] + acc[f][j];
  }
  conv_store<PF, CF, S, ACT>(acc, s_bias, mask, y16, y32, n, cy * TH, cx * TW, H, W, Cout, co0, vec);
}

// wt[ci][t'][co] = w[co][8 - t][ci]: the data gradient of a periodic 3x3
// convolution is the convolution of the output gradient with these weights
__global__ void k_flip(const bf16* __restrict__ w, bf16* __restrict__ wt, int32_t Cin, int32_t Cout) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)Cin * 9 * Cout) return;
  const int32_t co = (int32_t)(i % Cout), t = (int32_t)((i / Cout) % 9), ci = (int32_t)(i / (9 * (int64_t)Cout));
  wt[i] = w[((int64_t)co * 9 + (8 - t)) * Cin + ci];
}

// ---------------------------------------------------------------------------
// Weight and bias gradients: dW[co][t][ci] = sum_p dY[p][co] X[p + s_t][ci],
// db[co] = sum_p dY[p][co].  Rows = output channels, columns = input
// channels of one tap, reduction over pixels, 32 of a row at a time
// (v_mfma_f32_32x32x16_bf16: a wave alone on its SIMD issues them at the full
// rate, 32 clocks each; of the 16x16x32 form one every 27 clocks, not 16).
//
// A wave owns a 32 (co) x 32 (ci) block of all nine taps and walks units: R
// rows of one 32-pixel column strip of one image (the last strip of a row may
// be narrower).  Per dY row y it needs the X rows y - 1, y, y + 1, whose
// fragments at the three column shifts stay in registers, so every X and dY
// value is loaded once per strip and passes through LDS once.  Both lie there
// as loaded (a pixel's 32 channels, 64 bytes) and ds_read_b64_tr_b16 hands
// each lane four pixels of one channel: a shift is a row offset, and the 32
// lanes that are served together read 256 consecutive bytes.
//
// The four waves of a workgroup take different units of one block and share
// nothing until the end, where their sums are added through LDS: no barrier in
// the loop, and a quarter of the partials.  A wave has its SIMD to itself: the
// accumulators, four rows of loads in flight and the next row's fragments,
// read while this one's MFMAs run, take ~370 registers.  Partials go to
// `part`, [chunk][block][tap, quarter][lane][4] and the block's 32 bias sums;
// k_wgrad_sum adds the chunks in a fixed order.  With one chunk (`dw` given)
// the sums are the result.  Cin % 8 == Cout % 8 == 0.
//
// Bound: MFMA and LDS, 0.5 us a row of 32 pixels in short launches (the MFMAs
// alone 0.34), memory for 32 channels at 256^2 (67 MB at 8 TB/s from the
// last-level cache).  With k_wgrad_sum, against a kernel whose workgroups
// shared 32 x 32 blocks over a barrier a row and transposed in two-byte stores
// (1024 of them, 38 MB of partials), and one tap a workgroup for rows that are
// not whole strips (us, batch 8): 64 -> 64 at 128^2 28.1 -> 19.6; 32 -> 32 at
// 256^2 31.6 -> 21.0; 128 -> 128 at 64^2 30.5 -> 21.6; 256 -> 192 at 16^2 30.6
// -> 16.0; 128 -> 128 at 50 x 60 68.0 -> 20.7; 32 -> 32 at 200 x 230, batch 3,
// 110.6 -> 17.0.  Eight rows of loads in flight took 1 to 3 us longer.
// ---------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWgradPart = 9 * 32 * 32 + 32;      // floats of a block's partials
constexpr int kWgradWave = (48 + 32) * 32;        // LDS elements of a wave: X row (34 pixels of 48), dY row
constexpr int kWgradRed = 4 * 9 * 4 * 64 * 16;    // LDS bytes: the waves' sums, which overlay the rows
constexpr int kWgradLds = kWgradRed + 4 * 32 * 4; // and their bias sums

// four results of a lane to dw: D rows (co) = 8 quarter + 4 (lane / 32) + e,
// column (ci) = lane % 32
__device__ __forceinline__ void wgrad_put(float* __restrict__ dw, f32x4 v, int32_t t, int32_t quarter, int32_t lane,
                                          int32_t coB, int32_t ciB, int32_t Cin, int32_t Cout) {
  const int32_t co = coB + 8 * quarter + 4 * (lane >> 5), ci = ciB + (lane & 31);
  if (ci >= Cin) return;
#pragma unroll
  for (int e = 0; e < 4; e++)
    if (co + e < Cout) dw[((int64_t)(co + e) * 9 + t) * Cin + ci] = v[e];
}

template <bool RAG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_wgrad(
    const bf16* __restrict__ x, const bf16* __restrict__ dy, float* __restrict__ part, float* __restrict__ dw,
    float* __restrict__ db, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t R, uint32_t units, uint32_t per,
    int32_t nblk) {
  constexpr int D = 4;  // rows of loads in flight
  extern __shared__ __attribute__((aligned(16))) char s_wg[];
  const int32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this workgroup's (chunk, block): each XCD (workgroup b runs on XCD b % 8)
  // takes a contiguous range, so that the blocks of one chunk share its L2
  const uint32_t nb = gridDim.x, b = blockIdx.x, q8 = nb / 8, r8 = nb % 8, xcd = b % 8;
  const uint32_t lin = xcd * q8 + (xcd < r8 ? xcd : r8) + b / 8;
  const int32_t chunk = (int32_t)(lin / (uint32_t)nblk), blk = (int32_t)lin - chunk * nblk;
  const int32_t nci = (Cin + 31) / 32;
  const int32_t ciB = (blk % nci) * 32, coB = (blk / nci) * 32;
  const uint32_t segs = (uint32_t)(W + 31) / 32, cps = (uint32_t)(H + R - 1) / (uint32_t)R;

  bf16* s_x = (bf16*)s_wg + wave * kWgradWave;
  bf16* s_d = s_x + 48 * 32;
  const int32_t at = 8 * lane;  // item lane + 64 h of a row: pixel, channel group
  // a lane's part of a transposing read: pixel 8 (lane / 32) + lane % 16 / 4
  // (+ 4, + 16), channels 16 (lane / 16 % 2) + 4 (lane % 4) ..
  const int32_t tr = (8 * (lane >> 5) + ((lane & 15) >> 2)) * 32 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  auto frag = [&](const bf16* p) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(p + 4 * 32));
    return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // orders a wave's own LDS accesses (other lanes') for the compiler; the
  // hardware keeps a wave's LDS accesses in order
  auto fence = [&]() __attribute__((always_inline)) { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  const int64_t xrow = (int64_t)W * Cin, drow = (int64_t)W * Cout;
  constexpr uint32_t kBad = 0xffffffffu;  // past any row: reads zero
  auto fetch = [&](const bf16* row, uint32_t off) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)row, (short)0, (int)0xffffffff, 0x00020000);
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
  };

  // a unit: its loads' offsets in a row (what lies outside the strip or the
  // channels reads as zero), its rows, and the first rows' loads
  uint32_t xo[3], dof[2], keep[2][4];
  int32_t rows = 0, yx = 0, yd = 0;
  const bf16 *xim = x, *dim = dy, *xp = x, *dp = dy;
  struct Row {
    u32x4 x[3], d[2];
  } ring[D], first, second;
  // the next X and dY rows; both run on past the unit's last row (around the
  // image: in bounds, and not used)
  auto load_x = [&](Row& r) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 3; h++) r.x[h] = fetch(xp, xo[h]);
    yx = yx + 1 == H ? 0 : yx + 1;
    xp = yx ? xp + xrow : xim;
  };
  auto load_d = [&](Row& r) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) r.d[h] = fetch(dp, dof[h]);
    yd = yd + 1 == H ? 0 : yd + 1;
    dp = yd ? dp + drow : dim;
  };
  auto begin = [&](uint32_t u) __attribute__((always_inline)) {
    const uint32_t rest = u / cps, n = rest / segs;
    const int32_t y0 = (int32_t)(u - rest * cps) * R, x0 = (int32_t)(rest - n * segs) * 32;
    const int32_t w = W - x0 < 32 ? W - x0 : 32;
    rows = R < H - y0 ? R : H - y0;
#pragma unroll
    for (int h = 0; h < 3; h++) {
      const int32_t c = (lane >> 2) + 16 * h, ch = ciB + 8 * (lane & 3);
      xo[h] = c <= w + 1 && ch < Cin ? (uint32_t)(wrapi(x0 + c - 1, W) * (int64_t)Cin + ch) * 2 : kBad;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int32_t c = (lane >> 2) + 16 * h, ch = coB + 8 * (lane & 3);
      dof[h] = c < w && ch < Cout ? (uint32_t)((x0 + c) * (int64_t)Cout + ch) * 2 : kBad;
      // the strip's pixels among a lane's fragment elements
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int32_t p = 16 * h + 8 * (lane >> 5) + 2 * e;
        keep[h][e] = (p < w ? 0xffffu : 0u) | (p + 1 < w ? 0xffff0000u : 0u);
      }
    }
    xim = x + (int64_t)n * H * xrow;
    dim = dy + (int64_t)n * H * drow;
    yx = y0 > 0 ? y0 - 1 : H - 1;
    yd = y0;
    xp = xim + yx * xrow;
    dp = dim + yd * drow;
    load_x(first);
    load_x(second);
    load_x(ring[0]);
    load_d(ring[0]);
#pragma unroll
    for (int k = 1; k < D; k++) {
      load_x(ring[k]);
      load_d(ring[k]);
    }
  };
  auto store_x = [&](const Row& r) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 3; h++) *(u32x4*)&s_x[at + 512 * h] = r.x[h];
  };
  // bias sums: channels 8 (lane % 4) .. of this lane's pixels
  float bsum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  auto store_d = [&](const Row& r) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      *(u32x4*)&s_d[at + 512 * h] = r.d[h];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        bsum[2 * e] += __builtin_bit_cast(float, r.d[h][e] << 16);
        bsum[2 * e + 1] += __builtin_bit_cast(float, r.d[h][e] & 0xffff0000u);
      }
    }
  };
  // fragments (16 pixels each): dY rows s, s + 1; X rows s .. s + 3 at the
  // three column shifts
  u32x4 fa[2][2], fb[4][3][2];
  auto read_x = [&](u32x4 (*bb)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int h = 0; h < 2; h++) bb[d][h] = frag(s_x + tr + (16 * h + d) * 32);
  };
  auto read_d = [&](u32x4* a) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) a[h] = frag(s_d + tr + 16 * h * 32);
  };
  // a narrow strip: zero against zero past its last pixel, whatever X holds
  auto clip = [&](u32x4 (*bb)[2]) __attribute__((always_inline)) {
    if (!RAG) return;
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) bb[d][h][e] &= keep[h][e];
  };
  f32x16 acc[9];
  // dY row s against X rows s, s + 1, s + 2, while the next rows go from
  // registers through LDS to fragments
  auto step = [&](int v, bool more) __attribute__((always_inline)) {
    if (more) {
      fence();
      store_x(ring[(v + 1) % D]);
      store_d(ring[(v + 1) % D]);
      fence();
      load_x(ring[(v + 1) % D]);
      load_d(ring[(v + 1) % D]);
    }
    clip(fb[(v + 2) & 3]);
    if (more) {
      read_x(fb[(v + 3) & 3]);
      read_d(fa[(v + 1) & 1]);
    }
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[v & 1][h]),
                                                         __builtin_bit_cast(bf16x8, fb[(v + t / 3) & 3][t % 3][h]),
                                                         acc[t], 0, 0, 0);
  };

  uint32_t u = ((uint32_t)chunk * 4 + wave) * per;
  const uint32_t u1 = u + per < units ? u + per : units;
  if (u < u1) begin(u);
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[t][e] = 0.0f;
  while (u < u1) {
    fence();
    store_x(first);
    fence();
    read_x(fb[0]);
    fence();
    store_x(second);
    fence();
    read_x(fb[1]);
    fence();
    store_x(ring[0]);
    store_d(ring[0]);
    fence();
    load_x(ring[0]);
    load_d(ring[0]);
    read_x(fb[2]);
    read_d(fa[0]);
    clip(fb[0]);
    clip(fb[1]);
    int32_t s = 0;
    for (; s + D < rows; s += D) {
#pragma unroll
      for (int v = 0; v < D; v++) step(v, true);
    }
    const int32_t left = rows - s;  // 1 .. D
#pragma unroll
    for (int v = 0; v < D; v++)
      if (v < left) step(v, v + 1 < left);
    if (++u < u1) begin(u);
  }

  // the four waves' sums, added in wave order
  float* out = part + ((int64_t)chunk * nblk + blk) * kWgradPart;
  f32x4* red = (f32x4*)s_wg;
  float* s_bias = (float*)(s_wg + kWgradRed);
#pragma unroll
  for (int e = 0; e < 8; e++) {  // over the 16 lanes of a channel group
#pragma unroll
    for (int m = 4; m < 64; m *= 2) bsum[e] += __shfl_xor(bsum[e], m);
  }
  if (lane < 4) {
#pragma unroll
    for (int e = 0; e < 8; e++) s_bias[wave * 32 + 8 * lane + e] = bsum[e];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int q = 0; q < 4; q++)
      red[(wave * 36 + t * 4 + q) * 64 + lane] =
          (f32x4){acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const int32_t f = 4 * k + wave;
    f32x4 v = red[f * 64 + lane];
#pragma unroll
    for (int j = 1; j < 4; j++) v += red[(j * 36 + f) * 64 + lane];
    if (dw) {
      wgrad_put(dw, v, k, wave, lane, coB, ciB, Cin, Cout);
    } else {
      *(f32x4*)(out + (f * 64 + lane) * 4) = v;
    }
  }
  if (tid < 32) {
    const float v = s_bias[tid] + s_bias[32 + tid] + s_bias[64 + tid] + s_bias[96 + tid];
    if (!dw) out[9 * 32 * 32 + tid] = v;
    else if (db && ciB == 0 && coB + tid < Cout) db[coB + tid] = v;
  }
}

// dw and db (optional) from k_wgrad's partials, the chunks added in a fixed
// order: a workgroup takes 1024 / NG consecutive floats of a block; its NG
// groups of threads read them as 16-byte runs from every NG-th chunk (group q:
// chunks q, q + NG, ...), and the groups' sums are added in group order.
template <int NG>
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* __restrict__ part, float* __restrict__ dw,
                                                   float* __restrict__ db, int32_t Cin, int32_t Cout, int32_t nblk,
                                                   int32_t nparts) {
  constexpr int TG = 256 / NG, kTiles = (kWgradPart / 4 + TG - 1) / TG;
  __shared__ f32x4 s_sum[NG][TG];
  const int32_t tid = threadIdx.x, c = tid % TG, q = tid / TG;
  const int32_t blk = (int32_t)blockIdx.x / kTiles, at = ((int32_t)blockIdx.x % kTiles) * TG + c;
  const int64_t stride = (int64_t)nblk * kWgradPart;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  if (4 * at < kWgradPart) {
    const float* p = part + (int64_t)blk * kWgradPart + 4 * at;
    int32_t k = q;
    // eight chunks' loads in flight per step; the adds stay in chunk order
    for (; k + 7 * NG < nparts; k += 8 * NG) {
      f32x4 v[8];
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = *(const f32x4*)(p + (int64_t)(k + i * NG) * stride);
#pragma unroll
      for (int i = 0; i < 8; i++) acc += v[i];
    }
    for (; k < nparts; k += NG) acc += *(const f32x4*)(p + (int64_t)k * stride);
  }
  s_sum[q][c] = acc;
  __syncthreads();
  if (q != 0 || 4 * at >= kWgradPart) return;
#pragma unroll
  for (int i = 1; i < NG; i++) acc += s_sum[i][c];
  const int32_t nci = (Cin + 31) / 32, ciB = (blk % nci) * 32, coB = (blk / nci) * 32;
  if (at >= 9 * 256) {
    const int32_t co = coB + 4 * at - 9 * 32 * 32;
    if (db && ciB == 0) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (co + e < Cout) db[co + e] = acc[e];
    }
    return;
  }
  wgrad_put(dw, acc, at / 256, at / 64 % 4, at % 64, coB, ciB, Cin, Cout);
}

// ---------------------------------------------------------------------------
// Weight and bias gradients of small layers.  k_wgrad's fixed costs (three X
// rows before the first product, the waves' sums through LDS, partials of whole
// 32 x 32 blocks) are most of its time there: 10.8 us for 32 -> 32 at 64^2,
// batch 1, where k_wgrad_rows takes 9.3, and 12.5 for 192 -> 256 at 4^2, batch
// 8, where k_wgrad_flat takes 11.1 (wgrad_plan chooses).
//
// k_wgrad_flat: a workgroup (4 waves) owns a 64 (co) x 64 (ci) block of one
// tap and a chunk of the flattened batch's pixels; per step of 32 pixels every
// thread loads one 16-byte run of dY (8 channels of a pixel) and one of the
// tap-shifted X, and stores them channel-major into LDS (double buffered: the
// next step's runs are loaded while the waves run the current MFMAs); each wave
// accumulates a 32 x 32 sub-block.  The workgroups of tap 4 (no shift) and the
// first ci block also sum their dY runs for the bias.  Each chunk writes its
// partial block to `part` ([chunk][Cout * 9 * Cin + Cout]); k_reduce_parts adds
// the chunks in a fixed order, so the result is deterministic.  Maps of a few
// pixels waste no lanes on rows shorter than a strip.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_wgrad_flat(const bf16* __restrict__ x, const bf16* __restrict__ dy,
                                                    float* __restrict__ part, int32_t N, int32_t H, int32_t W,
                                                    int32_t Cin, int32_t Cout, int32_t chunk) {
  constexpr int LD = 40;
  __shared__ __attribute__((aligned(16))) bf16 s_dy[2][64 * LD];  // [co][pixel]
  __shared__ __attribute__((aligned(16))) bf16 s_x[2][64 * LD];   // [ci][pixel]
  __shared__ float s_b[32][65];                                    // bias partials [pixel lane][co]
  const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t cit = (Cin + 63) / 64;
  int32_t bq = blockIdx.y;
  const int32_t t = bq % 9;
  bq /= 9;
  const int32_t ciB = (bq % cit) * 64, coB = (bq / cit) * 64;
  const bool do_bias = t == 4 && ciB == 0;
  const int64_t npix = (int64_t)N * H * W;
  const int64_t p0 = (int64_t)blockIdx.x * chunk;
  const int64_t pend = p0 + chunk < npix ? p0 + chunk : npix;
  const int32_t dyo = t / 3 - 1, dxo = t % 3 - 1;
  // loader: pixel q of the step, channel group gg (8 channels)
  const int32_t q = tid >> 3, gg = tid & 7;
  const int32_t co_ld = coB + 8 * gg, ci_ld = ciB + 8 * gg;
  const bool co_ok = co_ld < Cout, ci_ok = ci_ld < Cin;
  const bf16x8 zero = {};
  bf16x8 rdy, rx;
  float bsum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  auto load = [&](int64_t q0) __attribute__((always_inline)) {
    const int64_t p = q0 + q;
    rdy = zero;
    rx = zero;
    if (p < pend) {
      if (co_ok) rdy = *(const bf16x8*)(dy + p * Cout + co_ld);
      if (ci_ok) {
        const int32_t xx = (int32_t)(p % W);
        const int64_t r = p / W;
        const int32_t yy = (int32_t)(r % H);
        const int64_t im = r / H;
        const int32_t sy = wrapi(yy + dyo, H), sx = wrapi(xx + dxo, W);
        rx = *(const bf16x8*)(x + ((im * H + sy) * W + sx) * Cin + ci_ld);
      }
    }
  };
  auto store = [&](int32_t buf) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      s_dy[buf][(8 * gg + e) * LD + q] = rdy[e];
      s_x[buf][(8 * gg + e) * LD + q] = rx[e];
    }
    if (do_bias) {
#pragma unroll
      for (int e = 0; e < 8; e++) bsum[e] += bf2f(rdy[e]);
    }
  };
  // consumer: wave (wave / 2, wave % 2) owns co rows 32 * (wave / 2) .., ci 32 * (wave % 2) ..
  const int32_t wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
  const int32_t kq = 8 * (lane >> 4), rl = lane & 15;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  load(p0);
  store(0);
  __syncthreads();
  int32_t buf = 0;
  for (int64_t q0 = p0; q0 < pend; q0 += 32) {
    const bool more = q0 + 32 < pend;
    if (more) load(q0 + 32);
    bf16x8 a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; i++) a[i] = *(const bf16x8*)&s_dy[buf][(wr + 16 * i + rl) * LD + kq];
#pragma unroll
    for (int j = 0; j < 2; j++) b[j] = *(const bf16x8*)&s_x[buf][(wc + 16 * j + rl) * LD + kq];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    if (more) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  const int64_t nw = (int64_t)Cout * 9 * Cin;
  float* out = part + (int64_t)blockIdx.x * (nw + Cout);
  // D rows (co) = wr + 16 i + 4 (lane / 16) + e, column (ci) = wc + 16 j + lane % 16
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int32_t ci = ciB + wc + 16 * j + rl;
    if (ci >= Cin) continue;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int32_t co = coB + wr + 16 * i + 4 * (lane >> 4) + e;
        if (co < Cout) out[((int64_t)co * 9 + t) * Cin + ci] = acc[i][j][e];
      }
  }
  if (do_bias) {  // the 32 pixel lanes' sums per channel, added in a fixed order
#pragma unroll
    for (int e = 0; e < 8; e++) s_b[q][8 * gg + e] = bsum[e];
    __syncthreads();
    if (tid < 64) {
      float sb = 0.0f;
      for (int k = 0; k < 32; k++) sb += s_b[k][tid];
      if (coB + tid < Cout) out[nw + coB + tid] = sb;
    }
  }
}

// k_wgrad_rows (W % 32 == 0): a workgroup owns a 32 (co) x 32 (ci) block of all
// nine taps and walks R rows of one 32-pixel column strip of one image.  Per
// row y it loads the dY row (32 pixels x CB) and the X row y + 1 (34 pixels,
// x0 - 1 .. x0 + 32, periodic); X rows y - 1, y, y + 1 stay in a four-row LDS
// ring.  LDS rows are channel-major (pixels contiguous, the MFMA's k), 40
// elements a row, with the 8-pixel blocks of columns 0..31 permuted per row
// (block ^ (row / 8) % 4) so that the transposing two-byte stores of eight
// channel rows fall in different banks.  The tap shift dx = -1, 0, +1 is a B
// operand read at column offset 0, 1, 2: one aligned 16-byte read plus the next
// dword, shifted by one element with v_alignbit for the odd offset.  Waves tile
// the block 2 x 2; the workgroups of the first ci block also sum the dY rows
// for the bias.  Partials as k_wgrad_flat's: of the layer's channels, not of
// whole blocks.
__device__ __forceinline__ int32_t wg_col(int32_t row, int32_t c) { return c < 32 ? c ^ (8 * ((row >> 3) & 3)) : c; }

__global__ __launch_bounds__(256) void k_wgrad_rows(const bf16* __restrict__ x, const bf16* __restrict__ dy,
                                                    float* __restrict__ part, int32_t N, int32_t H, int32_t W,
                                                    int32_t Cin, int32_t Cout, int32_t R) {
  constexpr int CB = 32, IB = 32;  // channels of a block
  constexpr int LD = 40;
  constexpr int TI = CB / 32, TJ = IB / 32;  // 16 x 16 tiles per wave along co and ci
  constexpr int DG = CB / 8, XG = IB / 8;    // 16-byte channel groups of a pixel
  constexpr int XITEMS = 34 * XG;            // X row loads (pixel, group)
  __shared__ __attribute__((aligned(16))) bf16 s_x[4][IB * LD];
  __shared__ __attribute__((aligned(16))) bf16 s_dy[2][CB * LD];
  __shared__ float s_b[32][CB + 1];
  const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t segs = W / 32, cps = (H + R - 1) / R;
  const int32_t chunk = blockIdx.x;
  const int32_t rc = chunk % cps, sg = (chunk / cps) % segs, n = chunk / (cps * segs);
  const int32_t nci = (Cin + IB - 1) / IB;
  const int32_t ciB = (int32_t)(blockIdx.y % nci) * IB, coB = (int32_t)(blockIdx.y / nci) * CB;
  const int32_t y0 = rc * R, rows = R < H - y0 ? R : H - y0, x0 = sg * 32;
  const bool do_bias = ciB == 0;
  const bf16x8 zero = {};

  // dY loads: thread -> (pixel dpx, group dg), groups fastest (coalesced)
  const bool dy_item = tid < 32 * DG;
  const int32_t dpx = tid / DG, dg = tid % DG;
  const bool dy_ok = dy_item && coB + 8 * dg < Cout;
  const int64_t dy_col = (int64_t)(x0 + dpx) * Cout + coB + 8 * dg;
  // X loads: items tid and tid + 256 -> (column c, group g)
  int32_t xc[2], xg[2];
  bool xok[2], xitem[2];
  int64_t xcol[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int32_t u = tid + 256 * h;
    xitem[h] = u < XITEMS;
    xc[h] = u / XG;
    xg[h] = u % XG;
    xok[h] = xitem[h] && ciB + 8 * xg[h] < Cin;
    xcol[h] = (int64_t)wrapi(x0 + xc[h] - 1, W) * Cin + ciB + 8 * xg[h];
  }
  const int64_t img = (int64_t)n * H;

  struct Regs {
    bf16x8 d, xa, xb;
  };
  // the loads of X row k (image row y0 - 1 + k) and dY row y
  auto load = [&](int32_t k, int32_t y, bool with_dy) __attribute__((always_inline)) {
    Regs r;
    const int64_t xrow = (img + wrapi(y0 - 1 + k, H)) * W * Cin;
    r.xa = xok[0] ? *(const bf16x8*)(x + xrow + xcol[0]) : zero;
    r.xb = xok[1] ? *(const bf16x8*)(x + xrow + xcol[1]) : zero;
    r.d = (with_dy && dy_ok) ? *(const bf16x8*)(dy + (img + y) * W * Cout + dy_col) : zero;
    return r;
  };
  float bsum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  auto store_x = [&](const Regs& r, int32_t slot) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (!xitem[h]) continue;
      const bf16x8 v = h == 0 ? r.xa : r.xb;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int32_t row = 8 * xg[h] + e;
        s_x[slot][row * LD + wg_col(row, xc[h])] = v[e];
      }
    }
  };
  auto store_dy = [&](const Regs& r, int32_t slot) __attribute__((always_inline)) {
    if (!dy_item) return;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int32_t row = 8 * dg + e;
      s_dy[slot][row * LD + wg_col(row, dpx)] = r.d[e];
    }
    if (do_bias) {
#pragma unroll
      for (int e = 0; e < 8; e++) bsum[e] += bf2f(r.d[e]);
    }
  };

  const int32_t wr = (CB / 2) * (wave >> 1), wc = (IB / 2) * (wave & 1);
  const int32_t kq = 8 * (lane >> 4), rl = lane & 15;
  f32x4 acc[9][TI][TJ];
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int j = 0; j < TJ; j++) acc[t][i][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

  // prologue: X rows y0 - 1, y0, y0 + 1 and dY row y0, all loads in flight together
  {
    const Regs r0 = load(0, y0, true), r1 = load(1, y0, false), r2 = load(2, y0, false);
    store_x(r0, 0);
    store_x(r1, 1);
    store_x(r2, 2);
    store_dy(r0, 0);
  }
  __syncthreads();
  for (int32_t s = 0; s < rows; s++) {
    const bool more = s + 1 < rows;
    Regs nx;
    if (more) nx = load(s + 3, y0 + s + 1, true);
    const int32_t ds = s & 1;
    bf16x8 a[TI];
#pragma unroll
    for (int i = 0; i < TI; i++) {
      const int32_t row = wr + 16 * i + rl;
      a[i] = *(const bf16x8*)&s_dy[ds][row * LD + wg_col(row, kq)];
    }
#pragma unroll
    for (int dyi = 0; dyi < 3; dyi++) {
      const bf16* xr = s_x[(s + dyi) & 3];
#pragma unroll
      for (int j = 0; j < TJ; j++) {
        const int32_t row = wc + 16 * j + rl;
        const u32x4 v0 = *(const u32x4*)&xr[row * LD + wg_col(row, kq)];
        const uint32_t v1 = *(const uint32_t*)&xr[row * LD + wg_col(row, kq + 8)];
        const u32x4 vm = v0;  // columns kq .. kq + 7: pixel x + dx for dx = -1
        const u32x4 vz = {__builtin_amdgcn_alignbit(v0[1], v0[0], 16), __builtin_amdgcn_alignbit(v0[2], v0[1], 16),
                          __builtin_amdgcn_alignbit(v0[3], v0[2], 16), __builtin_amdgcn_alignbit(v1, v0[3], 16)};
        const u32x4 vp = {v0[1], v0[2], v0[3], v1};
        const bf16x8 bm = __builtin_bit_cast(bf16x8, vm), bz = __builtin_bit_cast(bf16x8, vz),
                     bp = __builtin_bit_cast(bf16x8, vp);
#pragma unroll
        for (int i = 0; i < TI; i++) {
          acc[3 * dyi + 0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bm, acc[3 * dyi + 0][i][j], 0, 0, 0);
          acc[3 * dyi + 1][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bz, acc[3 * dyi + 1][i][j], 0, 0, 0);
          acc[3 * dyi + 2][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bp, acc[3 * dyi + 2][i][j], 0, 0, 0);
        }
      }
    }
    if (more) {
      store_x(nx, (s + 3) & 3);
      store_dy(nx, ds ^ 1);
    }
    __syncthreads();
  }

  const int64_t nw = (int64_t)Cout * 9 * Cin;
  float* out = part + (int64_t)chunk * (nw + Cout);
  // D rows (co) = wr + 16 i + 4 (lane / 16) + e, column (ci) = wc + 16 j + lane % 16
#pragma unroll
  for (int j = 0; j < TJ; j++) {
    const int32_t ci = ciB + wc + 16 * j + rl;
    if (ci >= Cin) continue;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int32_t co = coB + wr + 16 * i + 4 * (lane >> 4) + e;
        if (co >= Cout) continue;
#pragma unroll
        for (int t = 0; t < 9; t++) out[((int64_t)co * 9 + t) * Cin + ci] = acc[t][i][j][e];
      }
  }
  if (do_bias) {  // the 32 pixel columns' sums per channel, added in a fixed order
    if (dy_item) {
#pragma unroll
      for (int e = 0; e < 8; e++) s_b[dpx][8 * dg + e] = bsum[e];
    }
    __syncthreads();
    if (tid < CB) {
      float sb = 0.0f;
      for (int k = 0; k < 32; k++) sb += s_b[k][tid];
      if (coB + tid < Cout) out[nw + coB + tid] = sb;
    }
  }
}

// dw[i] (i < nw) and db[i - nw] (nw <= i < nw + Cout, when db is given):
// the chunks' partials added in a fixed order.  A workgroup takes 64
// consecutive entries; its 16 groups of 16 threads read them as float4 runs
// from every 16th chunk (group g: chunks g, g + 16, ...), and the groups'
// sums are added in group order.  Rows are nw + Cout floats, a multiple of
// 8 (Cin % 8 == Cout % 8 == 0), so the runs are aligned.
__global__ __launch_bounds__(256) void k_reduce_parts(const float* __restrict__ part, float* __restrict__ dw,
                                                      float* __restrict__ db, int64_t nw, int32_t Cout,
                                                      int32_t nparts) {
  __shared__ float s_sum[16][65];
  const int32_t tid = threadIdx.x, c4 = tid & 15, g = tid >> 4;
  const int64_t stride = nw + Cout;
  const int64_t n = db ? stride : nw;
  const int64_t i0 = (int64_t)blockIdx.x * 64 + 4 * c4;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  if (i0 < n) {
    const float* p = part + i0;
    int32_t k = g;
    // four chunks' loads in flight per step; the adds stay in chunk order
    for (; k + 48 < nparts; k += 64) {
      const f32x4 v0 = *(const f32x4*)(p + (int64_t)k * stride);
      const f32x4 v1 = *(const f32x4*)(p + (int64_t)(k + 16) * stride);
      const f32x4 v2 = *(const f32x4*)(p + (int64_t)(k + 32) * stride);
      const f32x4 v3 = *(const f32x4*)(p + (int64_t)(k + 48) * stride);
      acc += v0;
      acc += v1;
      acc += v2;
      acc += v3;
    }
    for (; k < nparts; k += 16) acc += *(const f32x4*)(p + (int64_t)k * stride);
  }
#pragma unroll
  for (int e = 0; e < 4; e++) s_sum[g][4 * c4 + e] = acc[e];
  __syncthreads();
  if (tid < 64) {
    const int64_t i = (int64_t)blockIdx.x * 64 + tid;
    if (i < n) {
      float s = 0.0f;
#pragma unroll
      for (int q = 0; q < 16; q++) s += s_sum[q][tid];
      if (i < nw) dw[i] = s;
      else db[i - nw] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// Elementwise, pooling, resampling
// ---------------------------------------------------------------------------
// g16 = bf16(g32 * (y > 0)) (ReLU gradient through the layer output), or
// just the conversion when y is null
__global__ void k_relu_grad(const float* __restrict__ g32, const bf16* __restrict__ y, bf16* __restrict__ g16,
                            int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float g = g32[i];
  if (y && !(bf2f(y[i]) > 0.0f)) g = 0.0f;
  g16[i] = f2bf(g);
}

// g16 *= (y > 0), in place
__global__ void k_relu_mask(bf16* __restrict__ g16, const bf16* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  if (!(bf2f(y[i]) > 0.0f)) g16[i] = f2bf(0.0f);
}

__global__ void k_add(const bf16* __restrict__ a, const bf16* __restrict__ b, bf16* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  out[i] = f2bf(bf2f(a[i]) + bf2f(b[i]));
}

// 2x2 average pool (H, W even), NHWC
__global__ void k_pool2(const bf16* __restrict__ x, bf16* __restrict__ y, int32_t N, int32_t H, int32_t W, int32_t C) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int32_t h = H / 2, w = W / 2;
  if (i >= (int64_t)N * h * w * C) return;
  const int32_t c = (int32_t)(i % C);
  const int64_t q = i / C;
  const int32_t xx = (int32_t)(q % w), yy = (int32_t)((q / w) % h);
  const int64_t im = q / ((int64_t)w * h);
  const int64_t b = ((im * H + 2 * yy) * W + 2 * xx) * C + c;
  const float s = bf2f(x[b]) + bf2f(x[b + C]) + bf2f(x[b + (int64_t)W * C]) + bf2f(x[b + (int64_t)W * C + C]);
  y[i] = f2bf(0.25f * s);
}

// gradient of the pool: every input pixel gets a quarter of its output's
__global__ void k_pool2_grad(const bf16* __restrict__ dy, bf16* __restrict__ dx, int32_t N, int32_t H, int32_t W,
                             int32_t C) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * H * W * C) return;
  const int32_t c = (int32_t)(i % C);
  const int64_t q = i / C;
  const int32_t xx = (int32_t)(q % W), yy = (int32_t)((q / W) % H);
  const int64_t im = q / ((int64_t)W * H);
  dx[i] = f2bf(0.25f * bf2f(dy[((im * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c]));
}

// nearest 2x upsampling of x [N][h][w][C] into [N][2h][2w][C]
__global__ void k_up2(const bf16* __restrict__ x, bf16* __restrict__ y, int32_t N, int32_t h, int32_t w, int32_t C) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int32_t H = 2 * h, W = 2 * w;
  if (i >= (int64_t)N * H * W * C) return;
  const int32_t c = (int32_t)(i % C);
  const int64_t q = i / C;
  const int32_t xx = (int32_t)(q % W), yy = (int32_t)((q / W) % H);
  const int64_t im = q / ((int64_t)W * H);
  y[i] = x[((im * h + yy / 2) * w + xx / 2) * C + c];
}

// its gradient: the sum over each 2x2 block
__global__ void k_up2_grad(const bf16* __restrict__ dy, bf16* __restrict__ dx, int32_t N, int32_t h, int32_t w,
                           int32_t C) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * h * w * C) return;
  const int32_t c = (int32_t)(i % C);
  const int64_t q = i / C;
  const int32_t xx = (int32_t)(q % w), yy = (int32_t)((q / w) % h);
  const int64_t im = q / ((int64_t)w * h);
  const int32_t W = 2 * w;
  const int64_t b = ((im * 2 * h + 2 * yy) * W + 2 * xx) * C + c;
  const float s = bf2f(dy[b]) + bf2f(dy[b + C]) + bf2f(dy[b + (int64_t)W * C]) + bf2f(dy[b + (int64_t)W * C + C]);
  dx[i] = f2bf(s);
}

// ---------------------------------------------------------------------------
// Fused passes of the skip connections, 8 channels (16 bytes) a thread
// (C % 8 == 0); each rounds to bf16 where the unfused sequence of the
// kernels above does, so the results are the same bits.
// ---------------------------------------------------------------------------
// out = bf16(up2(x) + skip): x [N][h][w][C] upsampled (nearest) and added
// to skip [N][2h][2w][C] (k_up2 then k_add)
__global__ void k_up2_add(const bf16* __restrict__ x, const bf16* __restrict__ skip, bf16* __restrict__ out,
                          int32_t N, int32_t h, int32_t w, int32_t C) {
  const int32_t C8 = C / 8, H = 2 * h, W = 2 * w;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * H * W * C8) return;
  const int32_t c = 8 * (int32_t)(i % C8);
  const int64_t q = i / C8;
  const int32_t xx = (int32_t)(q % W), yy = (int32_t)((q / W) % H);
  const int64_t im = q / ((int64_t)W * H);
  const bf16x8 a = *(const bf16x8*)(x + ((im * h + yy / 2) * w + xx / 2) * C + c);
  const bf16x8 b = *(const bf16x8*)(skip + q * C + c);
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] = f2bf(bf2f(a[e]) + bf2f(b[e]));
  *(bf16x8*)(out + q * C + c) = r;
}

// dx = bf16(bf16(dy / 4 upsampled) + skip), zero where mask <= 0 (mask
// optional): the pool's gradient plus the skip connection's, through the
// ReLU of the pooled layer (k_pool2_grad, k_add, k_relu_mask)
__global__ void k_pool2_grad_add(const bf16* __restrict__ dy, const bf16* __restrict__ skip,
                                 const bf16* __restrict__ mask, bf16* __restrict__ dx, int32_t N, int32_t H,
                                 int32_t W, int32_t C) {
  const int32_t C8 = C / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * H * W * C8) return;
  const int32_t c = 8 * (int32_t)(i % C8);
  const int64_t q = i / C8;
  const int32_t xx = (int32_t)(q % W), yy = (int32_t)((q / W) % H);
  const int64_t im = q / ((int64_t)W * H);
  const bf16x8 d = *(const bf16x8*)(dy + ((im * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c);
  const bf16x8 sk = *(const bf16x8*)(skip + q * C + c);
  bf16x8 m = {};
  if (mask) m = *(const bf16x8*)(mask + q * C + c);
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    bf16 v = f2bf(bf2f(f2bf(0.25f * bf2f(d[e]))) + bf2f(sk[e]));
    if (mask && !(bf2f(m[e]) > 0.0f)) v = f2bf(0.0f);
    r[e] = v;
  }
  *(bf16x8*)(dx + q * C + c) = r;
}

// dx = bf16(sum of dy over each 2x2 block), zero where mask <= 0 (mask
// optional): up2's gradient through the ReLU of the layer below
// (k_up2_grad, k_relu_mask)
__global__ void k_up2_grad_mask(const bf16* __restrict__ dy, const bf16* __restrict__ mask, bf16* __restrict__ dx,
                                int32_t N, int32_t h, int32_t w, int32_t C) {
  const int32_t C8 = C / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * h * w * C8) return;
  const int32_t c = 8 * (int32_t)(i % C8);
  const int64_t q = i / C8;
  const int32_t xx = (int32_t)(q % w), yy = (int32_t)((q / w) % h);
  const int64_t im = q / ((int64_t)w * h);
  const int32_t W = 2 * w;
  const int64_t b = ((im * 2 * h + 2 * yy) * W + 2 * xx) * C + c;
  const bf16x8 d0 = *(const bf16x8*)(dy + b), d1 = *(const bf16x8*)(dy + b + C);
  const bf16x8 d2 = *(const bf16x8*)(dy + b + (int64_t)W * C), d3 = *(const bf16x8*)(dy + b + (int64_t)W * C + C);
  bf16x8 m = {};
  if (mask) m = *(const bf16x8*)(mask + q * C + c);
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    bf16 v = f2bf(bf2f(d0[e]) + bf2f(d1[e]) + bf2f(d2[e]) + bf2f(d3[e]));
    if (mask && !(bf2f(m[e]) > 0.0f)) v = f2bf(0.0f);
    r[e] = v;
  }
  *(bf16x8*)(dx + q * C + c) = r;
}

// 2x2 average pool, 8 channels a thread (k_pool2's arithmetic)
__global__ void k_pool2_v8(const bf16* __restrict__ x, bf16* __restrict__ y, int32_t N, int32_t H, int32_t W,
                           int32_t C) {
  const int32_t C8 = C / 8, h = H / 2, w = W / 2;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * h * w * C8) return;
  const int32_t c = 8 * (int32_t)(i % C8);
  const int64_t q = i / C8;
  const int32_t xx = (int32_t)(q % w), yy = (int32_t)((q / w) % h);
  const int64_t im = q / ((int64_t)w * h);
  const int64_t b = ((im * H + 2 * yy) * W + 2 * xx) * C + c;
  const bf16x8 a0 = *(const bf16x8*)(x + b), a1 = *(const bf16x8*)(x + b + C);
  const bf16x8 a2 = *(const bf16x8*)(x + b + (int64_t)W * C), a3 = *(const bf16x8*)(x + b + (int64_t)W * C + C);
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] = f2bf(0.25f * (bf2f(a0[e]) + bf2f(a1[e]) + bf2f(a2[e]) + bf2f(a3[e])));
  *(bf16x8*)(y + q * C + c) = r;
}

// loss = sum over pixels and the first `used` of C channels of
// (pred - target)^2 / count; grad = 2 (pred - target) / count (0 elsewhere).
// Per-block partial sums of the loss.
__global__ void k_mse(const float* __restrict__ pred, const float* __restrict__ target, float* __restrict__ grad,
                      bf16* __restrict__ grad16, float* __restrict__ part, int64_t npix, int32_t C, int32_t used,
                      float inv_count) {
  __shared__ float s[256];
  const int32_t t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * 256;
  const int64_t i = base + t;
  // pixel and channel of i from the block's (one wave-uniform 64-bit divide)
  // and 32-bit arithmetic
  const int64_t pb = base / C;
  const int32_t r = (int32_t)(base - pb * C) + t;
  float l = 0.0f;
  if (i < npix * C) {
    const int32_t c = r % C;
    float g = 0.0f;
    if (c < used) {
      const float d = pred[i] - target[(pb + r / C) * used + c];
      l = d * d * inv_count;
      g = 2.0f * d * inv_count;
    }
    if (grad) grad[i] = g;
    if (grad16) grad16[i] = f2bf(g);
  }
  // the block's sum as a binary tree over its 256 threads (thread t adds
  // t + k for k = 128, 64, ..., 1); the levels below 64 run in wave 0 with
  // shuffles, which pair the same lanes, so the sum is the same bits
  s[t] = l;
  __syncthreads();
  if (t < 128) s[t] += s[t + 128];
  __syncthreads();
  if (t < 64) {
    float v = s[t] + s[t + 64];
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) v += __shfl_down(v, k, 64);
    if (t == 0) part[blockIdx.x] = v;
  }
}

// Adam on FP32 master weights, with the BF16 copy the convolutions read
__global__ void k_adam(float* __restrict__ w, bf16* __restrict__ w16, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (w16) w16[i] = f2bf(wi);
}

// Adam over many tensors in one launch: element i of the concatenation lies
// in the segment k with seg[k].off <= i < seg[k].off + seg[k].n (binary
// search over the nseg offsets).  The arithmetic is k_adam's; a segment
// with wt16 is a convolution's [Cout][9][Cin] weights whose flipped bf16
// copy (k_flip's layout) is written beside w16.
// hyper (optional): lr, c1, c2 read from device memory instead of the
// arguments, so that a captured graph serves every step
__global__ void k_adam_multi(const swe_nn_adam_seg* __restrict__ seg, int32_t nseg, int64_t total, float lr,
                             float b1, float b2, float eps, float c1, float c2, const float* __restrict__ hyper) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  if (hyper) {
    lr = hyper[0];
    c1 = hyper[1];
    c2 = hyper[2];
  }
  // the segment of the block's first element (a wave-uniform search), then
  // advanced for lanes past its end (a block meets few segments)
  const int64_t i0 = (int64_t)blockIdx.x * 256;
  int32_t lo = 0, hi = nseg - 1;
  while (lo < hi) {
    const int32_t mid = (lo + hi + 1) >> 1;
    if (seg[mid].off <= i0) lo = mid;
    else hi = mid - 1;
  }
  while (lo + 1 < nseg && seg[lo + 1].off <= i) ++lo;
  const swe_nn_adam_seg& sg = seg[lo];
  const int64_t j = i - sg.off;
  const float gi = sg.g[j];
  const float mi = b1 * sg.m[j] + (1.0f - b1) * gi;
  const float vi = b2 * sg.v[j] + (1.0f - b2) * gi * gi;
  sg.m[j] = mi;
  sg.v[j] = vi;
  const float wi = sg.w[j] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  sg.w[j] = wi;
  if (sg.w16) ((bf16*)sg.w16)[j] = f2bf(wi);
  if (sg.wt16) {
    // j = (co * 9 + t) * cin + ci; 32-bit division where the segment allows
    // (a 64-bit divide per element cost more than the update's memory traffic)
    int32_t ci, t, co;
    if (sg.n <= 0x7fffffffLL) {
      const uint32_t ju = (uint32_t)j, cin = (uint32_t)sg.cin, q = ju / cin;
      ci = (int32_t)(ju - q * cin);
      t = (int32_t)(q % 9u);
      co = (int32_t)(q / 9u);
    } else {
      ci = (int32_t)(j % sg.cin);
      t = (int32_t)((j / sg.cin) % 9);
      co = (int32_t)(j / (9 * (int64_t)sg.cin));
    }
    ((bf16*)sg.wt16)[((int64_t)ci * 9 + (8 - t)) * sg.cout + co] = f2bf(wi);
  }
}

// ---------------------------------------------------------------------------
// Input features of the surrogate, computed in float from the float maps and
// rounded to bf16 only at the end (the map's slopes are far below the bf16
// resolution of the heights themselves): x[n][y][x][0..7] = height anomaly,
// sediment, cos and sin of the wind azimuth, periodic central differences
// along the two map axes, the periodic 5-point Laplacian, 0.
// ---------------------------------------------------------------------------
__global__ void k_features(const float* __restrict__ h, const float* __restrict__ s, const float* __restrict__ mean,
                           const float* __restrict__ az, int32_t N, int32_t H, int32_t W, float h_scale,
                           float s_scale, float g_scale, float l_scale, bf16* __restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)N * H * W) return;
  const int32_t xx = (int32_t)(i % W), yy = (int32_t)((i / W) % H);
  const int64_t n = i / ((int64_t)W * H);
  const float* hn = h + n * H * W;
  const float c = hn[(int64_t)yy * W + xx];
  const float up = hn[(int64_t)wrapi(yy + 1, H) * W + xx], dn = hn[(int64_t)wrapi(yy - 1, H) * W + xx];
  const float rt = hn[(int64_t)yy * W + wrapi(xx + 1, W)], lt = hn[(int64_t)yy * W + wrapi(xx - 1, W)];
  bf16x8 v;
  v[0] = f2bf((c - mean[n]) / h_scale);
  v[1] = f2bf(s ? s[i] / s_scale : 0.0f);
  v[2] = f2bf(cosf(az[n]));
  v[3] = f2bf(sinf(az[n]));
  v[4] = f2bf(0.5f * (up - dn) / g_scale);
  v[5] = f2bf(0.5f * (rt - lt) / g_scale);
  v[6] = f2bf(((up + dn) + (rt + lt) - 4.0f * c) / l_scale);
  v[7] = f2bf(0.0f);
  *(bf16x8*)(x + i * 8) = v;
}

// ---------------------------------------------------------------------------
// Fixed-point mass projection: the predicted change d (float, per cell) is
// turned into int64 units of 2^-32 whose sum is exactly `target`: q_i =
// round(d_i * 2^32 * scale) and the residual target - sum(q) spread as evenly
// as integers allow (the first r cells get one unit more), then added to the
// master.
// ---------------------------------------------------------------------------
// one cell's predicted change in units of 2^-32, |q| < 2^62 (NaN -> 0)
__device__ __forceinline__ int64_t fx_units(float d, float scale) {
  float v = rintf(d * scale * 4294967296.0f);
  v = v > 4.0e18f ? 4.0e18f : (v < -4.0e18f ? -4.0e18f : v);
  return v == v ? (int64_t)v : 0;
}

__global__ void k_fx_sum(const float* __restrict__ d, int64_t n, float scale, int64_t* __restrict__ part) {
  __shared__ int64_t s[256];
  int64_t acc = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    acc += fx_units(d[i], scale);
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

__global__ void k_fx_apply(const float* __restrict__ d, int64_t n, float scale, const int64_t* __restrict__ part,
                           int32_t nparts, int64_t target, int64_t* __restrict__ master) {
  int64_t sum = 0;
  for (int32_t k = 0; k < nparts; k++) sum += part[k];
  const int64_t resid = target - sum;
  // resid = qq * n + rr with 0 <= rr < n
  int64_t qq = resid / n, rr = resid % n;
  if (rr < 0) {
    rr += n;
    qq -= 1;
  }
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    master[i] += fx_units(d[i], scale) + qq + (i < rr ? 1 : 0);
}

}  // namespace swenn

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
using namespace swenn;

static inline hipStream_t S(void* s) { return (hipStream_t)s; }
static inline unsigned G(int64_t n) { return (unsigned)((n + 255) / 256); }
#define SWENN_LAUNCH_CHECK() return hipGetLastError() == hipSuccess ? 0 : -2

extern "C" {

// Layers of few input channels on maps of whole 32-pixel strips
static bool conv_rows(int32_t W, int32_t Cin, int32_t Cout, int64_t P) {
  return W % 32 == 0 && (Cin <= 32 || (Cin <= 64 && (int64_t)Cout * P <= ((int64_t)1 << 23)));
}

// Slices of a split reduction: layers whose grid of 128-pixel blocks has fewer
// workgroups than the chip has CUs, ~768 over the slices, >= 8 steps of 32
// channels each, at most 8.  The tile kernels sum the slices in one workgroup
// (they need no workspace), but a layer given the workspace keeps the slices'
// order of additions.
static int32_t conv_slices(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout) {
  const int64_t P = (int64_t)N * H * W;
  if (conv_rows(W, Cin, Cout, P)) return 1;
  const int64_t mt = (P + 127) / 128;
  const int32_t nt = Cout <= 16 ? 16 : (Cout <= 32 ? 32 : (Cout <= 64 || mt * ((Cout + 127) / 128) < 512 ? 64 : 128));
  const int64_t wgs = mt * ((Cout + nt - 1) / nt), ksteps = 9 * ((Cin + 31) / 32);
  if (wgs >= 256 || ksteps < 24) return 1;
  int64_t z = (768 + wgs - 1) / wgs;
  if (z > ksteps / 8) z = ksteps / 8;
  if (z > 8) z = 8;
  return z < 2 ? 1 : (int32_t)z;
}

// The shape of a layer's workgroups (k_conv_tile up to 32 input channels,
// k_conv_wide above)
struct ConvTile {
  int32_t pf, cf, s, per;
  int64_t wgs;
  int32_t kc, two;
  size_t lds;
};
static bool conv_tile(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t kz, ConvTile* t) {
  const int32_t segs = (W + 15) / 16;
  t->s = segs % 2 == 0 ? 2 : 1;
  auto tiles = [&](int32_t pf) {
    const int32_t th = 4 * pf / t->s;
    return (int64_t)N * ((H + th - 1) / th) * (segs / t->s);
  };
  auto wgs = [&](int32_t pf, int32_t cf) { return tiles(pf) * ((Cout + 16 * cf - 1) / (16 * cf)); };
  t->kc = t->two = 0;
  t->lds = 0;
  const bool wide = Cin > 32;
  if (!wide) {
    // the largest workgroups that still make enough of them for the chip's 256
    // CUs, which hold two to four each (32 -> 64 at 128^2, batch 8: (4, 4)
    // 11.4 us, (2, 4) 11.9, (2, 2) 11.7; 32 -> 32 at 256^2, batch 1, (4, 2)
    // 9.5, (2, 2) 9.7, (1, 2) 10.1)
    struct Shape {
      int32_t pf, cf, wgs;
    };
    static const Shape k16[] = {{4, 1, 0}};
    static const Shape k32[] = {{4, 2, 512}, {2, 2, 192}, {1, 2, 0}};
    static const Shape k64[] = {{4, 4, 512}, {2, 4, 400}, {2, 2, 192}, {1, 2, 0}};
    const Shape* sh = Cout <= 16 ? k16 : (Cout <= 32 ? k32 : k64);
    while (wgs(sh->pf, sh->cf) < sh->wgs) sh++;
    t->pf = sh->pf;
    t->cf = sh->cf;
  } else {
    // The shape of least estimated time: rounds of workgroups (one or two to a
    // CU, by LDS) times a workgroup's fragment reads, PF + CF a k-step; two on
    // a CU take 1.3 times as long as one alone.  Measured (us) at batch 8: 192
    // -> 192 at 32^2, (4, 2) 17.7 (one round), (2, 4) 19.7 (one), (1, 2) 23.1
    // (two rounds of two), (2, 2) 25.5 (two); 128 -> 192 there, (2, 2) 13.3,
    // (4, 2) 14.8, (2, 4) 15.9; 128 -> 128 at 64^2, (2, 4) 18.2, (2, 2) 22.5,
    // (4, 2) 24.7; 256 -> 192 at 16^2, (1, 2) 13.9, (2, 2) 16.0, (2, 4) 23.8;
    // at batch 1 256 -> 256 at 16^2, (1, 1) 11.4, (1, 2) 13.4 (slices over
    // workgroups and a pass that adds them: 13.3).
    static const int32_t kShape[][2] = {{4, 4}, {4, 2}, {2, 4}, {2, 2}, {1, 2}, {1, 1}};
    double best = 0.0;
    for (const auto& sh : kShape) {
      const int32_t pf = sh[0], cf = sh[1], kmax = 32 * conv_wide_chunks(pf, cf);
      if ((cf > 2 && Cout <= 32) || (kz > 1 && pf * cf > 8)) continue;
      const int32_t kc = Cin > kmax ? kmax : (Cin + 31) / 32 * 32;
      const size_t rows = (size_t)(4 * pf / t->s + 2) * (16 * t->s + 2), row = (size_t)(kc + 8) * 2;
      const size_t one = (rows + 16 * cf) * row + 64 * cf, two = one + 16 * cf * row;
      if (one > 163840) continue;
      const int64_t w = wgs(pf, cf), per_cu = one <= 81920 ? 2 : 1;
      const double est = (double)((w + 256 * per_cu - 1) / (256 * per_cu)) * (pf + cf) * (per_cu == 2 && w > 256 ? 1.3 : 1.0);
      if (best > 0.0 && est >= best) continue;
      best = est;
      t->pf = pf;
      t->cf = cf;
      t->kc = kc;
      // a second weight buffer saves a barrier a tap; not at the price of the
      // second workgroup on a CU
      t->two = two <= 81920 || (per_cu == 1 && two <= 163840);
      t->lds = t->two ? two : one;
    }
    if (best == 0.0) return false;
  }
  const int64_t n = tiles(t->pf), ncob = (Cout + 16 * t->cf - 1) / (16 * t->cf);
  // one chunk: a workgroup keeps its weights over several tiles, one round of
  // workgroups in all
  const int64_t round = 256 * conv_tile_waves(t->pf, t->cf);
  t->per = !wide ? (int32_t)((n * ncob + round - 1) / round) : 1;
  t->wgs = (n + t->per - 1) / t->per * ncob;
  return t->wgs <= 0x7fffffffLL && n <= 0x3fffffffLL;
}

static int conv_launch(const void* x, int32_t N, int32_t H, int32_t W, int32_t Cin, const void* w, const float* bias,
                       int32_t Cout, int act, const void* mask, void* y16, float* y32, void* stream,
                       const float* work = nullptr, int64_t work_len = 0) {
  if (!x || !w || N < 1 || H < 1 || W < 1 || Cin < 8 || Cin % 8 || Cout < 1 || (!y16 && !y32)) return -1;
  const int64_t P = (int64_t)N * H * W;
  // the kernels' buffer loads take 32-bit byte offsets below 2^31
  if (P * Cin * 2 >= ((int64_t)1 << 31) || (int64_t)Cout * 9 * Cin * 2 >= ((int64_t)1 << 31)) return -1;
  // refused since these layers' 32-channel blocks were a grid's second axis
  // (the tile kernels have no such limit)
  if (conv_rows(W, Cin, Cout, P) && (Cout + 31) / 32 > 65535) return -1;
  const bf16* xx = (const bf16*)x;
  const bf16* ww = (const bf16*)w;
  const bf16* mm = (const bf16*)mask;
  bf16* yy = (bf16*)y16;
  int32_t kz = conv_slices(N, H, W, Cin, Cout);
  if (!work || work_len < (int64_t)kz * P * Cout) kz = 1;
  ConvTile ct;
  if (!conv_tile(N, H, W, Cin, Cout, kz, &ct)) return -1;
  // 16-byte stores and mask loads where every row of channels is aligned to them
  const int32_t vec = Cout % 8 == 0 && !(((uintptr_t)y16 | (uintptr_t)y32 | (uintptr_t)mask) & 15);
  const dim3 g((unsigned)ct.wgs);
#define SWENN_CT(PF_, CF_, S_, AC)                                                                               \
  hipLaunchKernelGGL((k_conv_tile<PF_, CF_, S_, AC>), g, dim3(256), 0, S(stream), xx, ww, bias, mm, yy, y32, N, H, \
                     W, Cin, Cout, ct.per, vec)
#define SWENN_CW_(PF_, CF_, S_, AC, SP_)                                                                          \
  hipLaunchKernelGGL((k_conv_wide<PF_, CF_, S_, AC, SP_>), g, dim3(256), ct.lds, S(stream), xx, ww, bias, mm, yy, \
                     y32, N, H, W, Cin, Cout, ct.kc, kz, ct.two, vec)
#define SWENN_CW(PF_, CF_, S_, AC) SWENN_CW_(PF_, CF_, S_, AC, false)
#define SWENN_CWS(PF_, CF_, S_, AC) SWENN_CW_(PF_, CF_, S_, AC, true)
#define SWENN_CT_ACT(K_, PF_, CF_, S_)    \
  if (act == 1) K_(PF_, CF_, S_, 1);      \
  else if (act == 2) K_(PF_, CF_, S_, 2); \
  else K_(PF_, CF_, S_, 0)
#define SWENN_CT_S(K_, PF_, CF_)                    \
  if (ct.s == 2) { SWENN_CT_ACT(K_, PF_, CF_, 2); } \
  else { SWENN_CT_ACT(K_, PF_, CF_, 1); }
  if (Cin > 32 && kz > 1) {
    if (ct.pf == 2 && ct.cf == 4) { SWENN_CT_S(SWENN_CWS, 2, 4); }
    else if (ct.pf == 4 && ct.cf == 2) { SWENN_CT_S(SWENN_CWS, 4, 2); }
    else if (ct.pf == 2 && ct.cf == 2) { SWENN_CT_S(SWENN_CWS, 2, 2); }
    else if (ct.cf == 2) { SWENN_CT_S(SWENN_CWS, 1, 2); }
    else { SWENN_CT_S(SWENN_CWS, 1, 1); }
  } else if (Cin > 32) {
    if (ct.pf == 4 && ct.cf == 4) { SWENN_CT_S(SWENN_CW, 4, 4); }
    else if (ct.pf == 2 && ct.cf == 4) { SWENN_CT_S(SWENN_CW, 2, 4); }
    else if (ct.pf == 4 && ct.cf == 2) { SWENN_CT_S(SWENN_CW, 4, 2); }
    else if (ct.pf == 2 && ct.cf == 2) { SWENN_CT_S(SWENN_CW, 2, 2); }
    else if (ct.cf == 2) { SWENN_CT_S(SWENN_CW, 1, 2); }
    else { SWENN_CT_S(SWENN_CW, 1, 1); }
  } else {
    if (ct.pf == 4 && ct.cf == 4) { SWENN_CT_S(SWENN_CT, 4, 4); }
    else if (ct.pf == 2 && ct.cf == 4) { SWENN_CT_S(SWENN_CT, 2, 4); }
    else if (ct.pf == 4 && ct.cf == 2) { SWENN_CT_S(SWENN_CT, 4, 2); }
    else if (ct.pf == 2 && ct.cf == 2) { SWENN_CT_S(SWENN_CT, 2, 2); }
    else if (ct.pf == 1 && ct.cf == 2) { SWENN_CT_S(SWENN_CT, 1, 2); }
    else { SWENN_CT_S(SWENN_CT, 4, 1); }
  }
#undef SWENN_CT_S
#undef SWENN_CT_ACT
#undef SWENN_CWS
#undef SWENN_CW
#undef SWENN_CW_
#undef SWENN_CT
  SWENN_LAUNCH_CHECK();
}

int64_t swe_nn_conv3x3_work(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout) {
  if (N < 1 || H < 1 || W < 1 || Cin < 1 || Cout < 1) return 0;
  const int32_t z = conv_slices(N, H, W, Cin, Cout);
  return z > 1 ? (int64_t)z * N * H * W * Cout : 0;
}

int swe_nn_conv3x3_ws(const void* x, int32_t N, int32_t H, int32_t W, int32_t Cin, const void* w, const float* bias,
                      int32_t Cout, int32_t act, const void* mask, void* y16, float* y32, float* work,
                      int64_t work_len, void* stream) {
  if (act < 0 || act > 2 || (act == 2 && !mask)) return -1;
  return conv_launch(x, N, H, W, Cin, w, bias, Cout, act, mask, y16, y32, stream, work, work_len);
}

int swe_nn_conv3x3(const void* x, int32_t N, int32_t H, int32_t W, int32_t Cin, const void* w, const float* bias,
                   int32_t Cout, int32_t relu, void* y16, float* y32, void* stream) {
  return conv_launch(x, N, H, W, Cin, w, bias, Cout, relu ? 1 : 0, nullptr, y16, y32, stream);
}

int swe_nn_conv3x3_masked(const void* x, int32_t N, int32_t H, int32_t W, int32_t Cin, const void* w,
                          const float* bias, int32_t Cout, const void* mask, void* y16, void* stream) {
  if (!y16) return -1;
  return conv_launch(x, N, H, W, Cin, w, bias, Cout, mask ? 2 : 0, mask, y16, nullptr, stream);
}

int swe_nn_flip(const void* w, int32_t Cin, int32_t Cout, void* wt, void* stream) {
  if (!w || !wt) return -1;
  hipLaunchKernelGGL(k_flip, dim3(G((int64_t)Cin * 9 * Cout)), dim3(256), 0, S(stream), (const bf16*)w, (bf16*)wt,
                     Cin, Cout);
  SWENN_LAUNCH_CHECK();
}

// How a weight gradient is split: 32 x 32 channel blocks, each over `chunks`
// workgroups of four waves with `per` units a wave.  One round of workgroups
// (a CU holds one), units as long as that allows (a unit loads two X rows more
// than it has), but of at least six rows: below, a wave's ~5 us outside its
// rows and the partials outweigh the 0.5 us a row.  Measured (us, with the pass
// over the partials) for a least of four / six / eight rows: 128 -> 192 at
// 32^2, batch 8, 16.8 / 16.6 / 15.9; 32 -> 32 at 200 x 230, batch 3, 17.8 /
// 17.0 / 16.1; 192 -> 256 at 12 x 16, batch 2, 11.9 / 10.1 / 9.8; the other
// way 32 -> 32 at 256^2, batch 1, 12.9 / 13.7 / 13.8; 64 -> 64 at 300 x 9,
// 14.2 / 15.0 / 15.2.  Chunks of at most eight rows in all become one, whose
// workgroups write the result: 256 -> 192 at 4^2, batch 2, 12.7 -> 9.5; to
// sixteen rows it loses (192 -> 256 at 8^2, batch 8, 14.6 -> 19.0).
//
// Small layers take the kernels above where those are estimated faster: times
// in us, fitted to 1,341 measured layers (two launches of a graph each; mean
// error 2% for k_wgrad and k_wgrad_rows, 5% for k_wgrad_flat), and only up to
// 13.5 (k_wgrad_flat 15), past which k_wgrad's rate decides.  Measured (small kernel / k_wgrad):
// 8 -> 32 at 128^2, batch 1, 9.5 / 12.1; 64 -> 32 there 11.5 / 12.6; 32 -> 32 at
// 256^2 14.2 / 13.7; 32 -> 64 at 4^2, batch 8, 8.6 / 12.1; 256 -> 256 at 4^2,
// batch 4, 10.2 / 9.4; 128 -> 192 at 8^2, batch 4, 13.3 / 12.4.
constexpr int32_t kWgradMinRows = 6, kWgradOneChunk = 8;
constexpr double kWgradSmallRows = 13.5, kWgradSmallFlat = 15.0;
enum WgradKind { kWgradStrips, kWgradRows, kWgradFlat };
struct WgradPlan {
  WgradKind kind;
  int32_t R;
  int64_t blocks, units, per, chunks;
  int64_t chunk;  // k_wgrad_flat: pixels
  int64_t work;   // floats of partials
};

// whole 32-pixel strips, R rows a workgroup (at least eight), ~1024 workgroups
static WgradPlan wgrad_rows_plan(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, double* us) {
  WgradPlan p{};
  p.kind = kWgradRows;
  p.blocks = (int64_t)((Cout + 31) / 32) * ((Cin + 31) / 32);
  const int64_t strips = (int64_t)N * (W / 32), cmax = (H + 7) / 8;
  int64_t cps = (1024 + strips * p.blocks - 1) / (strips * p.blocks);
  if (cps > cmax) cps = cmax;
  p.R = (int32_t)((H + cps - 1) / cps);
  p.chunks = strips * ((H + p.R - 1) / p.R);
  const double part = (double)Cout * (9.0 * Cin + 1.0) * 1e-6;  // partials of a chunk, millions
  p.work = p.chunks * ((int64_t)Cout * 9 * Cin + Cout);
  *us = 5.07 + 0.483 * p.R + 0.00397 * (double)(p.chunks * p.blocks) + 1.8 * (double)p.chunks * part +
        0.004 * (double)p.chunks;
  return p;
}

// flattened pixels, a multiple of 32 and at least 256 a workgroup, ~1024 workgroups
static WgradPlan wgrad_flat_plan(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, double* us) {
  WgradPlan p{};
  p.kind = kWgradFlat;
  p.blocks = (int64_t)((Cout + 63) / 64) * 9 * ((Cin + 63) / 64);
  const int64_t npix = (int64_t)N * H * W;
  p.chunk = ((npix * p.blocks + 1023) / 1024 + 31) / 32 * 32;
  if (p.chunk < 256) p.chunk = 256;
  p.chunks = (npix + p.chunk - 1) / p.chunk;
  const double part = (double)Cout * (9.0 * Cin + 1.0) * 1e-6, px = (double)(npix < p.chunk ? npix : p.chunk);
  p.work = p.chunks * ((int64_t)Cout * 9 * Cin + Cout);
  *us = 4.76 + 0.031 * px + (1.78 - 0.0028 * px) * part + 0.01315 * (double)(p.chunks * p.blocks) +
        1.17 * (double)p.chunks * part - (p.chunks > 1 ? 1.68 : 0.0);
  return p;
}

static WgradPlan wgrad_plan(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout) {
  WgradPlan p{};
  p.blocks = (int64_t)((Cout + 31) / 32) * ((Cin + 31) / 32);
  const int64_t strips = (int64_t)N * ((W + 31) / 32), waves = p.blocks >= 256 ? 4 : 4 * (256 / p.blocks);
  int64_t cps = waves / strips;
  const int64_t cmax = (H + kWgradMinRows - 1) / kWgradMinRows;
  if (cps > cmax) cps = cmax;
  if (cps < 1) cps = 1;
  p.R = (int32_t)((H + cps - 1) / cps);
  p.units = strips * ((H + p.R - 1) / p.R);
  p.per = (p.units + waves - 1) / waves;
  p.chunks = (p.units + 4 * p.per - 1) / (4 * p.per);
  // a few rows more a wave cost less than the pass that adds the chunks
  if (p.chunks * p.per * p.R <= kWgradOneChunk) {
    p.per *= p.chunks;
    p.chunks = 1;
  }
  p.work = p.chunks * p.blocks * kWgradPart;
  const double us = 5.90 + 0.432 * (double)p.R * (double)p.per + 1.04 * (double)(p.per - 1) +
                    (p.chunks > 1 ? 1.21 : 0.0) + 0.024 * (double)(p.chunks * p.blocks) - 0.0161 * (double)p.blocks +
                    0.30 * (double)(p.units < 4 ? p.units : 4);
  double small = 0.0;
  const WgradPlan q = W % 32 == 0 ? wgrad_rows_plan(N, H, W, Cin, Cout, &small) : wgrad_flat_plan(N, H, W, Cin, Cout, &small);
  // (k_wgrad counts units and addresses a row in 32 bits)
  const bool wide = p.units + 4 * p.per > 0xffffffffLL || (int64_t)W * (Cin > Cout ? Cin : Cout) * 2 >= 0xffffffffLL;
  return wide || (small < us && small < (W % 32 == 0 ? kWgradSmallRows : kWgradSmallFlat)) ? q : p;
}

int64_t swe_nn_wgrad_work(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout) {
  if (N < 1 || H < 1 || W < 1 || Cin < 1 || Cout < 1) return 0;
  return wgrad_plan(N, H, W, Cin, Cout).work;
}
int swe_nn_wgrad(const void* x, const void* dy, int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout,
                 float* dw, float* db, float* work, int64_t work_len, void* stream) {
  if (!x || !dy || !dw || !work || (uintptr_t)work % 16) return -1;
  if (N < 1 || H < 1 || W < 1 || Cin < 8 || Cout < 8 || Cin % 8 || Cout % 8) return -1;
  const WgradPlan p = wgrad_plan(N, H, W, Cin, Cout);
  if (work_len < p.work) return -1;
  // blocks a grid's second axis holds: 32 x 32, or 64 x 64 of one tap where a
  // row is not whole strips (k_wgrad has no such limit; refused all the same)
  const int64_t blocks = (int64_t)((Cout + 31) / 32) * ((Cin + 31) / 32);
  const int64_t tall = W % 32 ? (int64_t)((Cout + 63) / 64) * 9 * ((Cin + 63) / 64) : 0;
  if (blocks > 65535 || tall > 65535 || p.chunk > 0x7fffffffLL || p.chunks > 0x7fffffffLL / (p.kind == kWgradStrips ? p.blocks : 1))
    return -1;
  const bf16* xx = (const bf16*)x;
  const bf16* dd = (const bf16*)dy;
  if (p.kind != kWgradStrips) {
    const dim3 grid((unsigned)p.chunks, (unsigned)p.blocks);
    if (p.kind == kWgradRows)
      hipLaunchKernelGGL(k_wgrad_rows, grid, dim3(256), 0, S(stream), xx, dd, work, N, H, W, Cin, Cout, p.R);
    else
      hipLaunchKernelGGL(k_wgrad_flat, grid, dim3(256), 0, S(stream), xx, dd, work, N, H, W, Cin, Cout,
                         (int32_t)p.chunk);
    const int64_t nw = (int64_t)Cout * 9 * Cin, nred = db ? nw + Cout : nw;
    hipLaunchKernelGGL(k_reduce_parts, dim3((unsigned)((nred + 63) / 64)), dim3(256), 0, S(stream), work, dw, db, nw,
                       Cout, (int32_t)p.chunks);
    SWENN_LAUNCH_CHECK();
  }
  const dim3 grid((unsigned)(p.chunks * p.blocks));
  float* dw1 = p.chunks == 1 ? dw : nullptr;
  if (W % 32)
    hipLaunchKernelGGL(k_wgrad<true>, grid, dim3(256), kWgradLds, S(stream), xx, dd, work, dw1, db, H, W, Cin, Cout,
                       p.R, (uint32_t)p.units, (uint32_t)p.per, (int32_t)p.blocks);
  else
    hipLaunchKernelGGL(k_wgrad<false>, grid, dim3(256), kWgradLds, S(stream), xx, dd, work, dw1, db, H, W, Cin, Cout,
                       p.R, (uint32_t)p.units, (uint32_t)p.per, (int32_t)p.blocks);
  // one pass adds the chunks' weight and bias partials
  const int32_t nq = kWgradPart / 4;
  if (p.chunks >= 32)
    hipLaunchKernelGGL(k_wgrad_sum<16>, dim3((unsigned)(p.blocks * ((nq + 15) / 16))), dim3(256), 0, S(stream), work,
                       dw, db, Cin, Cout, (int32_t)p.blocks, (int32_t)p.chunks);
  else if (p.chunks > 1)
    hipLaunchKernelGGL(k_wgrad_sum<4>, dim3((unsigned)(p.blocks * ((nq + 63) / 64))), dim3(256), 0, S(stream), work,
                       dw, db, Cin, Cout, (int32_t)p.blocks, (int32_t)p.chunks);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_relu_grad(const float* g32, const void* y, void* g16, int64_t n, void* stream) {
  if (!g32 || !g16) return -1;
  hipLaunchKernelGGL(k_relu_grad, dim3(G(n)), dim3(256), 0, S(stream), g32, (const bf16*)y, (bf16*)g16, n);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_relu_mask(void* g16, const void* y, int64_t n, void* stream) {
  if (!g16 || !y) return -1;
  hipLaunchKernelGGL(k_relu_mask, dim3(G(n)), dim3(256), 0, S(stream), (bf16*)g16, (const bf16*)y, n);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_add(const void* a, const void* b, void* out, int64_t n, void* stream) {
  hipLaunchKernelGGL(k_add, dim3(G(n)), dim3(256), 0, S(stream), (const bf16*)a, (const bf16*)b, (bf16*)out, n);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_pool2(const void* x, void* y, int32_t N, int32_t H, int32_t W, int32_t C, void* stream) {
  if (!x || !y || H % 2 || W % 2) return -1;
  if (C % 8 == 0)
    hipLaunchKernelGGL(k_pool2_v8, dim3(G((int64_t)N * (H / 2) * (W / 2) * (C / 8))), dim3(256), 0, S(stream),
                       (const bf16*)x, (bf16*)y, N, H, W, C);
  else
    hipLaunchKernelGGL(k_pool2, dim3(G((int64_t)N * (H / 2) * (W / 2) * C)), dim3(256), 0, S(stream), (const bf16*)x,
                       (bf16*)y, N, H, W, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_up2_add(const void* x, const void* skip, void* out, int32_t N, int32_t h, int32_t w, int32_t C,
                   void* stream) {
  if (!x || !skip || !out || N < 1 || h < 1 || w < 1 || C < 8 || C % 8) return -1;
  hipLaunchKernelGGL(k_up2_add, dim3(G((int64_t)N * 4 * h * w * (C / 8))), dim3(256), 0, S(stream), (const bf16*)x,
                     (const bf16*)skip, (bf16*)out, N, h, w, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_pool2_grad_add(const void* dy, const void* skip, const void* mask, void* dx, int32_t N, int32_t H,
                          int32_t W, int32_t C, void* stream) {
  if (!dy || !skip || !dx || N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C < 8 || C % 8) return -1;
  hipLaunchKernelGGL(k_pool2_grad_add, dim3(G((int64_t)N * H * W * (C / 8))), dim3(256), 0, S(stream),
                     (const bf16*)dy, (const bf16*)skip, (const bf16*)mask, (bf16*)dx, N, H, W, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_up2_grad_mask(const void* dy, const void* mask, void* dx, int32_t N, int32_t h, int32_t w, int32_t C,
                         void* stream) {
  if (!dy || !dx || N < 1 || h < 1 || w < 1 || C < 8 || C % 8) return -1;
  hipLaunchKernelGGL(k_up2_grad_mask, dim3(G((int64_t)N * h * w * (C / 8))), dim3(256), 0, S(stream),
                     (const bf16*)dy, (const bf16*)mask, (bf16*)dx, N, h, w, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_pool2_grad(const void* dy, void* dx, int32_t N, int32_t H, int32_t W, int32_t C, void* stream) {
  if (H % 2 || W % 2) return -1;
  hipLaunchKernelGGL(k_pool2_grad, dim3(G((int64_t)N * H * W * C)), dim3(256), 0, S(stream), (const bf16*)dy,
                     (bf16*)dx, N, H, W, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_up2(const void* x, void* y, int32_t N, int32_t h, int32_t w, int32_t C, void* stream) {
  hipLaunchKernelGGL(k_up2, dim3(G((int64_t)N * 4 * h * w * C)), dim3(256), 0, S(stream), (const bf16*)x, (bf16*)y,
                     N, h, w, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_up2_grad(const void* dy, void* dx, int32_t N, int32_t h, int32_t w, int32_t C, void* stream) {
  hipLaunchKernelGGL(k_up2_grad, dim3(G((int64_t)N * h * w * C)), dim3(256), 0, S(stream), (const bf16*)dy, (bf16*)dx,
                     N, h, w, C);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_mse(const float* pred, const float* target, float* grad, void* grad16, float* part, int64_t npix,
               int32_t C, int32_t used, void* stream) {
  if (!pred || !target || !part || (!grad && !grad16) || npix < 1 || used < 1 || used > C) return -1;
  const float inv = 1.0f / (float)((double)npix * used);
  hipLaunchKernelGGL(k_mse, dim3(G(npix * C)), dim3(256), 0, S(stream), pred, target, grad, (bf16*)grad16, part, npix,
                     C, used, inv);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_adam(float* w, void* w16, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
                float eps, int32_t step, void* stream) {
  if (step < 1) return -1;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(G(n)), dim3(256), 0, S(stream), w, (bf16*)w16, g, m, v, n, lr, b1, b2, eps, c1, c2);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_adam_multi(const swe_nn_adam_seg* seg, int32_t nseg, int64_t total, float lr, float b1, float b2,
                      float eps, int32_t step, void* stream) {
  if (!seg || nseg < 1 || total < 0 || step < 1) return -1;
  if (total == 0) return 0;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam_multi, dim3(G(total)), dim3(256), 0, S(stream), seg, nseg, total, lr, b1, b2, eps, c1, c2,
                     (const float*)nullptr);
  SWENN_LAUNCH_CHECK();
}

void swe_nn_adam_hyper(float lr, float b1, float b2, int32_t step, float* out) {
  out[0] = lr;
  out[1] = 1.0f - powf(b1, (float)step);
  out[2] = 1.0f - powf(b2, (float)step);
}

int swe_nn_adam_multi_dev(const swe_nn_adam_seg* seg, int32_t nseg, int64_t total, const float* hyper, float b1,
                          float b2, float eps, void* stream) {
  if (!seg || !hyper || nseg < 1 || total < 0) return -1;
  if (total == 0) return 0;
  hipLaunchKernelGGL(k_adam_multi, dim3(G(total)), dim3(256), 0, S(stream), seg, nseg, total, 0.0f, b1, b2, eps, 0.0f,
                     0.0f, hyper);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_features(const float* h, const float* s, const float* mean, const float* az, int32_t N, int32_t H,
                    int32_t W, float h_scale, float s_scale, float g_scale, float l_scale, void* x, void* stream) {
  if (!h || !mean || !az || !x || N < 1 || H < 1 || W < 1) return -1;
  hipLaunchKernelGGL(k_features, dim3(G((int64_t)N * H * W)), dim3(256), 0, S(stream), h, s, mean, az, N, H, W,
                     h_scale, s_scale, g_scale, l_scale, (bf16*)x);
  SWENN_LAUNCH_CHECK();
}

int swe_nn_project_mass(const float* d, int64_t n, float scale, int64_t target, int64_t* master, int64_t* work,
                        void* stream) {
  if (!d || !master || !work || n < 1) return -1;
  const int32_t nparts = 256;
  hipLaunchKernelGGL(k_fx_sum, dim3(nparts), dim3(256), 0, S(stream), d, n, scale, work);
  hipLaunchKernelGGL(k_fx_apply, dim3(nparts), dim3(256), 0, S(stream), d, n, scale, (const int64_t*)work, nparts,
                     target, master);
  SWENN_LAUNCH_CHECK();
}

}  // extern "C"
