// HIP kernels of the warm-start network (gfx950): a 3-D U-Net over
// (space, space, time) patches, channels-last, BF16 activations and weights,
// FP32 accumulation, trained on the GPU by these kernels.
//
// Layouts (row-major, last index fastest):
//   activations  [n][d][h][w][c]  bf16 (c a multiple of 16)
//   weights      [27][co][ci]     bf16, tap = (kd * 3 + kh) * 3 + kw
//   masters      fp32 copies of the weights and biases, Adam moments
//
// 3x3x3 convolutions (stride 1, zero padding 1) are implicit GEMMs on the
// matrix cores: one wavefront computes 16 consecutive voxels along w by all
// output channels with v_mfma_f32_16x16x32_bf16 (M = voxels, N = 16 output
// channels, K = the 16 input channels of two taps per instruction). The input
// gradient is the same kernel run on the flipped, transposed weights; the
// weight gradient is a deterministic two-pass reduction (per-block FP32
// partial sums over voxel slabs, then a fixed-order sum).
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

#include "agd_launch.h"
#include "agdeblend_unet.h"

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// four biases, of any float pointer
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][8 (l / 16) + e] and
// B[8 (l / 16) + e][l % 16], e < 8, as 8 bf16 in a u32x4; D as for K = 16
__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

#define UT 256

static int hip_ok(hipError_t e, char const *what) {
  if (e != hipSuccess) {
    fprintf(stderr, "ERROR: HIP %s: %s\n", what, hipGetErrorString(e));
    return 1;
  }
  return 0;
}

static hipStream_t ustream(void *s) { return (hipStream_t)s; }

template <typename K, typename... A>
static int ulaunch(char const *name, K kernel, dim3 grid, dim3 block, void *stream,
                   A... args) {
  if (grid.x == 0 || grid.y == 0 || grid.z == 0) return 0;
  hipLaunchKernelGGL(kernel, grid, block, 0, ustream(stream), args...);
  return hip_ok(hipGetLastError(), name);
}

__device__ __forceinline__ float bf2f(uint16_t h) {
  return __uint_as_float((uint32_t)h << 16);
}
// round to nearest even: one v_cvt_pk_bf16_f32. (Rounded in integers, with the
// branch that keeps Inf and NaN, an output value cost some twenty
// instructions, more than its share of the matrix-core work: the inference
// pass's 16-channel layers issued five VALU instructions per matrix-core one.)
__device__ __forceinline__ uint16_t f2bf(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}

// ---------------------------------------------------------------------------
// Convolution (forward, or input gradient with flipped weights)
// ---------------------------------------------------------------------------
// Block tile: DB consecutive d planes x CT_H rows (h) x CT_W voxels (w) of
// one n, all output channels; one wave per row, 4 matrix-core tiles of 16
// voxels each. Per 16-channel input chunk the block stages that chunk of the
// weights ([27][CO][16]) once and walks the DB planes with a ring of three
// input planes in LDS ((CT_H + 2) rows x (CT_W + 2) voxels x 16 channels
// each; one new plane per step), so the input is read (DB + 2) / DB times
// instead of three. Each matrix-core step takes two taps: K = 32 is the 16
// channels of tap 2 s (lanes 0-31) and of tap 2 s + 1 (lanes 32-63), 14
// steps for the 27 taps (the last one's second tap has zero weights); both
// operands are 16-byte LDS reads per lane. Staging loads are branch-free
// (clamped address, zero selected afterwards) so a thread's loads stay in
// flight together.
// grid: (ceil(W / CT_W), ceil(H / CT_H), N * ceil(D / DB)); block 256.
// mode bits: 1 = add bias, 2 = ReLU on the output, 4 = multiply the output
// by (gate > 0) (the ReLU mask of the layer below, for input gradients).
#define CT_W 64
#define CT_H 4

// LDS rows of 16 bf16 channels (32 bytes) with their four 8-byte quarters
// rotated by (row >> 2) & 3: the 16 lanes of a matrix-core operand read
// (16 consecutive rows, one quarter) then fall in 16 distinct bank pairs
// instead of 4-way conflicts
__device__ __forceinline__ int swz_q(int row, int q) { return row * 16 + ((q ^ ((row >> 2) & 3)) << 2); }
__device__ __forceinline__ bf16x4 ld_swz(uint16_t const *base, int row, int q) {
  return *(bf16x4 const *)(base + swz_q(row, q));
}
// store 8 channels (quarters 2 half, 2 half + 1) of row
__device__ __forceinline__ void st_swz(uint16_t *base, int row, int half, uint4 v) {
  *(uint2 *)(base + swz_q(row, 2 * half)) = make_uint2(v.x, v.y);
  *(uint2 *)(base + swz_q(row, 2 * half + 1)) = make_uint2(v.z, v.w);
}
// The K = 32 operands read 16 bytes (8 channels, one half of a row) per
// lane. The LDS serves 128 bytes (32 banks) per cycle, i.e. 8 lanes of a
// 16-byte read: 8 consecutive rows of 32 bytes, one half each, span 256
// bytes, and rows r and r + 4 fall on the same banks; swapping the two
// halves of a row when (row >> 2) & 1 sends them to different banks, so
// every 8 lanes cover the 32 banks once
__device__ __forceinline__ int swz_h(int row, int half) {
  return row * 16 + ((half ^ ((row >> 2) & 1)) << 3);
}
__device__ __forceinline__ u32x4 ld_h(uint16_t const *base, int row, int half) {
  return *(u32x4 const *)(base + swz_h(row, half));
}
__device__ __forceinline__ void st_h(uint16_t *base, int row, int half, uint4 v) {
  *(uint4 *)(base + swz_h(row, half)) = v;
}

// byte offset of half `half` of row `row` (swz_h); adding a multiple of 8
// rows moves it by 32 bytes a row
__device__ __forceinline__ int off_h(int row, int half) {
  return row * 32 + ((half ^ ((row >> 2) & 1)) << 4);
}
__device__ __forceinline__ u32x4 ld_b(uint16_t const *base, int bytes) {
  return *(u32x4 const *)((char const *)base + bytes);
}
// four output channels of a voxel as bf16 (bias added; ReLU)
template <bool RELU>
__device__ __forceinline__ uint2 out4(f32x4 a, f32x4 b) {
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    v[r] = a[r] + b[r];
    if (RELU) v[r] = fmaxf(v[r], 0.f);
  }
  return make_uint2((uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                    (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16));
}

template <int CO, int CU, bool UPC = false>
struct ConvDepth {
  // depth planes per block: the ring saves input reads, the accumulators
  // (DB x 4 x CO / 16 tiles) cost registers
  static constexpr int DB = CO <= 16 ? ((CU && !UPC) ? 2 : 4) : (CO <= 32 ? 2 : 1);
};

// waves per SIMD the registers are bounded for: two where the LDS allows two
// blocks per CU, else one (the 64-channel layers, d2a on combined taps)
template <int CO, bool UPC>
struct ConvWaves {
  static constexpr int W = (CO >= 64 || (UPC && CO >= 32)) ? 1 : 2;
};

// Combined taps of a 3x3x3 convolution over a nearest x2 upsampled input.
// Along one axis, output index o = 2 c + p reads input o + k - 1 (k = 0, 1,
// 2), i.e. coarse c + floor((p + k - 1) / 2): for p = 0 the coarse offsets
// are -1 (k = 0) and 0 (k = 1, 2); for p = 1 they are 0 (k = 0, 1) and +1
// (k = 2). So per output parity the three taps become two, taps 0 and 1+2
// (p = 0) or 0+1 and 2 (p = 1), and the two read the input rows o - 1 + p
// and o + p. Applied along d and h (whose parities are uniform per plane
// and per row of a block), the 27 taps become 4 (a, b) pairs x 3 w taps for
// each of the 4 (pd, ph) parities: 48 combined taps, entry
// ((pd * 2 + ph) * 4 + a * 2 + b) * 3 + kw.

// CU > 0: the input is the concatenation [upsample(xu), x] without being
// formed: input channels [0, CU) are xu's ([n][D/2][H/2][W/2][CU], nearest
// x2 upsampling, D, H, W even) and [CU, CI) are x's ([n][D][H][W][CI - CU]).
// UPC: the xu channels use the 48 combined taps wcu ([48][CO][CU], built by
// k_up_weights from wt) instead of wt's 27: per 16-channel chunk 12
// combined taps, 6 matrix-core steps of two, instead of 27 taps in 14.
template <int CI, int CO, int CU, bool UPC = false>
__global__ __launch_bounds__(UT, (ConvWaves<CO, UPC>::W)) void k_conv3(
    uint16_t const *__restrict__ x, uint16_t const *__restrict__ xu,
    uint16_t const *__restrict__ wt, uint16_t const *__restrict__ wcu,
    float const *__restrict__ bias, uint16_t const *__restrict__ gate,
    uint16_t *__restrict__ y, uint16_t *__restrict__ pool, int D, int H, int W, int mode) {
  static_assert(CI % 16 == 0 && CO % 16 == 0 && CU % 16 == 0 && CU < CI,
                "channels in multiples of 16");
  static_assert(!UPC || CU > 0, "combined taps serve the upsampled channels");
  constexpr int CS = CI - CU;  // channels of x
  constexpr int NT = CO / 16;
  constexpr int DB = ConvDepth<CO, CU, UPC>::DB;
  constexpr int PW = CT_W + 2, PH = CT_H + 2;
  constexpr int PLANE = PH * PW * 16;  // bf16 elements of one staged plane
  constexpr int NPI = PH * PW * 2;     // staging items (8 channels) per plane
  constexpr int NWI = 27 * CO * 2;
  constexpr int NWU = 48 * CO * 2;     // staging items of the combined taps
  constexpr int NTW = UPC ? 48 : 28;   // taps the weight region holds (the 28th zero)
  constexpr int OBS = CO + 4;  // output staging row: CO channels + 4 (bank spread)
  // output staging: 4 x 64 rows of OBS, then the pooling partials [2][32][CO]
  constexpr int OSM = 4 * 64 * OBS + 2 * 32 * CO;
  constexpr int SMEM = 3 * PLANE + NTW * CO * 16 > OSM ? 3 * PLANE + NTW * CO * 16 : OSM;
  __shared__ __align__(16) uint16_t smem[SMEM];
  uint16_t *const sx = smem;               // ring of 3 input planes
  uint16_t *const sw = smem + 3 * PLANE;   // weights of the chunk
  int const tid = threadIdx.x;
  int const lane = tid & 63;
  int const wave = tid >> 6;
  int const ndb = (D + DB - 1) / DB;
  int const n = blockIdx.z / ndb;
  int const d0 = (blockIdx.z - n * ndb) * DB;
  int const h0 = blockIdx.y * CT_H;
  int const w0 = blockIdx.x * CT_W;
  // The weights are the matrix-core instruction's A operand and the voxels its
  // B, so that a lane ends with four neighbouring output channels of one
  // voxel: one 8-byte LDS write in the epilogue instead of four of 2.
  int const i = lane & 15;   // channel in the tile (weights), voxel (input, output)
  int const kq = lane >> 4;  // k group: channels 8 (kq & 1) .. + 7 of the step's tap kq >> 1
  // LDS byte offsets of the lane's operands, built once: the loop over the
  // taps then adds constants only. (Built at each step they were most of the
  // 6.4 vector instructions per matrix-core one, whose issue bounds these
  // layers: 96 -> 32 at 32 x 128 x 1024 960 us, now 846; the network on
  // 64 x 256 x 2048 5.04 ms, now 4.51; a step on 16 patches of 32 x 32 x 256
  // 4.19 ms, now 3.96.) Input: step st's tap 2 st + (kq >> 1) (the
  // 28th reads the 27th's voxels, with zero weights) within a plane of the
  // ring; weights: bof + 32 CO tap.
  constexpr int PLANEB = PH * PW * 32;
  constexpr bool STREAM = UPC && DB >= 4;
  constexpr int NST = STREAM ? 5 : 14;  // steps: positions of a plane, or taps
  int const hi = kq >> 1;
  int aof[NST];
#pragma unroll
  for (int st = 0; st < NST; ++st) {
    int const tl = 2 * st + hi, last = STREAM ? 8 : 26;
    int const t = (tl < last ? tl : last) % 9;
    aof[st] = off_h((wave + t / 3) * PW + i + t % 3, kq & 1);
  }
  int const bof = off_h(i, kq & 1) + hi * CO * 32;
  // ring slots (bytes) of the planes d0, d0 + 1, d0 + 2 modulo 3
  int const slot[3] = {d0 % 3 * PLANEB, (d0 + 1) % 3 * PLANEB, (d0 + 2) % 3 * PLANEB};
  if constexpr (!STREAM)  // the 28th tap (the combined taps come after it)
    for (int e = tid; e < CO * 2; e += UT)
      *(uint4 *)(sw + 27 * CO * 16 + e * 8) = make_uint4(0, 0, 0, 0);
  f32x4 acc[DB][4][NT];
#pragma unroll
  for (int j = 0; j < DB; ++j)
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[j][m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint16_t const *const xn = x + (int64_t)n * D * H * W * CS;
  int64_t const plane = (int64_t)H * W * CS;
  int const Hu = H / 2, Wu = W / 2;
  uint16_t const *const xun = CU ? xu + (int64_t)n * (D / 2) * Hu * Wu * CU : nullptr;
  int64_t const planeu = (int64_t)Hu * Wu * CU;
  constexpr int NPK = (NPI + UT - 1) / UT;  // staging items per thread and plane
  // per staging item: 32-bit offset within a plane (the same for every
  // plane and chunk) and whether its (h, w) lies inside the volume; items
  // past the last repeat it (same value, same place: no branch, so the
  // compiler keeps the loads ahead of the stores)
  uint32_t ioff[NPK], iofu[NPK];
  bool iok[NPK];
#pragma unroll
  for (int k = 0; k < NPK; ++k) {
    int const e0 = tid + k * UT;
    int const e = e0 < NPI ? e0 : NPI - 1;
    int const half = e & 1;
    int const r = e >> 1;
    int const pw = r % PW, ph = r / PW;
    int const hh = h0 + ph - 1, ww = w0 + pw - 1;
    iok[k] = hh >= 0 && hh < H && ww >= 0 && ww < W;
    ioff[k] = iok[k] ? (uint32_t)(hh * W + ww) * (uint32_t)CS + (uint32_t)(half * 8)
                     : (uint32_t)(half * 8);
    iofu[k] = iok[k] ? (uint32_t)((hh >> 1) * Wu + (ww >> 1)) * (uint32_t)CU + (uint32_t)(half * 8)
                     : (uint32_t)(half * 8);
  }
  // global loads of plane dd of chunk c, raw (clamped addresses) ...
  auto load_plane = [&](int dd, int c, uint4 (&v)[NPK]) {
    bool const okd = dd >= 0 && dd < D;
    bool const up = CU > 0 && c < CU / 16;  // the same for the whole block
    uint16_t const *const src = up ? xun + (okd ? dd >> 1 : 0) * planeu + c * 16
                                   : xn + (okd ? dd : 0) * plane + (c - CU / 16) * 16;
#pragma unroll
    for (int k = 0; k < NPK; ++k) v[k] = *(uint4 const *)(src + (up ? iofu[k] : ioff[k]));
  };
  // ... and their store into ring slot (dd + 3) % 3, zero outside the
  // volume (a mask, not a branch; applied here so that the loads stay in
  // flight until the store)
  auto store_plane = [&](int dd, uint4 const (&v)[NPK]) {
    bool const okd = dd >= 0 && dd < D;
    uint16_t *const dst = sx + ((dd + 3) % 3) * PLANE;
#pragma unroll
    for (int k = 0; k < NPK; ++k) {
      int const e0 = tid + k * UT;
      int const e = e0 < NPI ? e0 : NPI - 1;
      uint32_t const msk = (okd && iok[k]) ? ~0u : 0u;
      st_h(dst, e >> 1, e & 1, make_uint4(v[k].x & msk, v[k].y & msk, v[k].z & msk, v[k].w & msk));
    }
  };
  // a chunk's first three planes and its weights ([27][CO][16]), loaded
  // into registers (PRE: while the previous chunk is computed; for the
  // 64-channel layers, whose registers and LDS allow one block per CU
  // either way), then stored
  constexpr bool PRE = CO >= 64;
  constexpr int NXW = (NWI + UT - 1) / UT;
  uint4 xv[3][NPK], xw[NXW];
  auto load_chunk = [&](int c) {
#pragma unroll
    for (int q = 0; q < 3; ++q) load_plane(d0 - 1 + q, c, xv[q]);
#pragma unroll
    for (int k = 0; k < NXW; ++k) {
      int const e0 = tid + k * UT;
      int const e = e0 < NWI ? e0 : NWI - 1;
      xw[k] = *(uint4 const *)(wt + (int64_t)(e >> 1) * CI + c * 16 + (e & 1) * 8);  // tap * CO + co
    }
  };
  auto store_chunk = [&]() {
#pragma unroll
    for (int k = 0; k < NXW; ++k) {
      int const e0 = tid + k * UT;
      int const e = e0 < NWI ? e0 : NWI - 1;
      st_h(sw, e >> 1, e & 1, xw[k]);  // past the end: the last item again
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) store_plane(d0 - 1 + q, xv[q]);
  };
  // operands of one matrix-core step (two taps): A for the 4 voxel tiles,
  // B for the NT output channel tiles
  struct Ops {
    u32x4 a[4];
    u32x4 b[NT];
  };
  // UPC: the upsampled channels, on the 48 combined taps ([48][CO][CU]) and
  // staged at their own (coarse) resolution, the whole block's region at
  // once: coarse planes d0/2 - 1 .. (d0 + DB)/2, rows h0/2 - 1 ..
  // (h0 + CT_H)/2, columns w0/2 - 1 .. (w0 + CT_W)/2 (d0, h0, w0 even),
  // row (cd * CPH + ch) * CPW + cw of the ring's LDS. They are computed
  // after the x channels, whose last planes' compute overlaps the loads of
  // the first coarse chunk.
  constexpr int CPW = CT_W / 2 + 2, CPH = CT_H / 2 + 2, CPD = DB / 2 + 2;
  constexpr int NCI = CPD * CPH * CPW * 2;  // staging items (8 channels)
  constexpr int NCK = (NCI + UT - 1) / UT;
  static_assert(!UPC || (DB % 2 == 0 && CT_H % 2 == 0 && NCI * 8 <= 3 * PLANE),
                "coarse staging: whole coarse planes and rows, within the ring");
  static_assert(!UPC || NCK <= 32, "inside-the-volume bits of the coarse items");
  constexpr int NCW = (NWU + UT - 1) / UT;
  // per coarse item: its offset (the same for every chunk; 0 outside the
  // volume) and, in cok, whether it lies inside the volume
  int64_t coff[UPC ? NCK : 1];
  uint32_t cok = 0;
#pragma unroll
  for (int k = 0; k < (UPC ? NCK : 0); ++k) {
    int const e0 = tid + k * UT;
    int const e = e0 < NCI ? e0 : NCI - 1;
    int const half = e & 1, r = e >> 1;
    int const cw = r % CPW, t = r / CPW;
    int const gd = d0 / 2 - 1 + t / CPH, gh = h0 / 2 - 1 + t % CPH;
    int const gw = w0 / 2 - 1 + cw;
    bool const ok = gd >= 0 && gd < D / 2 && gh >= 0 && gh < Hu && gw >= 0 && gw < Wu;
    coff[k] = (ok ? (int64_t)gd * planeu + (int64_t)(gh * Wu + gw) * CU : 0) + half * 8;
    cok |= (ok ? 1u : 0u) << k;
  }
  // a coarse chunk's region, loaded into registers while the previous
  // chunk is computed (its combined weights, the same for every block,
  // come from L2 when stored)
  uint4 cv[UPC ? NCK : 1];
  auto load_coarse = [&](int c) {
#pragma unroll
    for (int k = 0; k < (UPC ? NCK : 0); ++k) cv[k] = *(uint4 const *)(xun + coff[k] + c * 16);
  };
  // the coarse chunks (UPC), chunk 0's region already in cv
  auto coarse_part = [&]() {
    if constexpr (UPC) {
#pragma unroll 1
      for (int c = 0; c < CU / 16; ++c) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NCW; ++k) {
          int const e0 = tid + k * UT;
          int const e = e0 < NWU ? e0 : NWU - 1;
          uint4 const v = *(uint4 const *)(wcu + (int64_t)(e >> 1) * CU + c * 16 + (e & 1) * 8);
          st_h(sw, e >> 1, e & 1, v);  // combined tap * CO + co
        }
#pragma unroll
        for (int k = 0; k < NCK; ++k) {
          int const e0 = tid + k * UT;
          int const e = e0 < NCI ? e0 : NCI - 1;
          uint32_t const msk = ((cok >> k) & 1u) ? ~0u : 0u;
          st_h(sx, e >> 1, e & 1,
               make_uint4(cv[k].x & msk, cv[k].y & msk, cv[k].z & msk, cv[k].w & msk));
        }
        __syncthreads();
        if (c + 1 < CU / 16) load_coarse(c + 1);
        __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the compute
        int const bofu = bof + ((h0 + wave) & 1) * 12 * CO * 32;
        static_assert(CPH * CPW % 8 == 0, "planes at whole swizzle periods");
        int cof[3];
#pragma unroll
        for (int sp = 0; sp < 3; ++sp) {
          int const u = 2 * sp + hi, b = u / 3, kw = u - 3 * b;
          cof[sp] = off_h(((wave + 1) / 2 + b) * CPW + 1 + ((i + kw - 1) >> 1), kq & 1);
        }
        // Streamed over the staged coarse planes: fine plane j (parity j & 1,
        // d0 even) reads coarse plane (j + 1) / 2 + a with its d-combination
        // a, so coarse plane cp feeds fine planes 2 (cp - a) - 1 and
        // 2 (cp - a) for a = 0, 1. Each A fragment (coarse plane cp, h
        // combination b, tap kw) is read once and used for those (up to
        // four) fine planes; K = 32 pairs two of the six (b, kw) positions.
        // Per fine plane the contributions keep their order (a = 0, then
        // a = 1; positions in order), so the sums are those of one plane at
        // a time.
#pragma unroll
        for (int cp = 0; cp < CPD; ++cp) {
#pragma unroll
          for (int sp = 0; sp < 3; ++sp) {
            // (b, kw) position 2 sp + hi of this lane: combined tap
            // (pd 2 + ph) 12 + a 6 + position
            u32x4 a4[4];
#pragma unroll
            for (int m = 0; m < 4; ++m)
              a4[m] = ld_b(sx, cof[sp] + cp * CPH * CPW * 32 + m * 8 * 32);
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
              for (int jp = 0; jp < 2; ++jp) {
                int const j = 2 * (cp - a) - 1 + jp;
                if (j >= 0 && j < DB) {
                  int const pd = j & 1;
#pragma unroll
                  for (int t = 0; t < NT; ++t) {
                    u32x4 const bt =
                        ld_b(sw, bofu + (pd * 24 + a * 6 + 2 * sp) * CO * 32 + t * 512);
#pragma unroll
                    for (int m = 0; m < 4; ++m) acc[j][m][t] = mfma32(bt, a4[m], acc[j][m][t]);
                  }
                }
              }
          }
        }
      }
    }
  };
  if constexpr (PRE) load_chunk(UPC ? CU / 16 : 0);
#pragma unroll 1
  for (int c = UPC ? CU / 16 : 0; c < CI / 16; ++c) {
    __syncthreads();
    if constexpr (!PRE) load_chunk(c);
    store_chunk();
    __syncthreads();
    // PRE: the next chunk's loads go out once this chunk's plane loads are
    // done (in the last plane steps), so that waiting for a plane never
    // waits for them
    bool const pre = PRE && c + 1 < CI / 16;
    if constexpr (STREAM) {
      // The x channels of d1a streamed over the input planes p = d0 - 1 ..
      // d0 + DB (in ring slot (p + 3) % 3): each A fragment (plane p, two
      // (kh, kw) positions of step s) is read once and used for the output
      // planes p + 1 - kd it feeds, with the weights of tap kd 9 + position
      // from LDS; plane p + 3 is loaded while plane p is computed and stored
      // into its slot.
#pragma unroll
      for (int jp = 0; jp < DB + 2; ++jp) {
        int const p = d0 - 1 + jp;
        uint4 nxt[NPK];
        bool const more = jp + 3 < DB + 2;  // plane p + 3 still an input
        if (more)
          load_plane(p + 3, c, nxt);
        else if (jp == DB - 1 && pre)
          load_chunk(c + 1);
        else if (jp == DB - 1 && c + 1 == CI / 16)
          load_coarse(0);
        __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the compute
#pragma unroll
        for (int st = 0; st < 5; ++st) {
          // position 2 st + hi; past the ninth: its voxels, zero weights
          unsigned const keep = st < 4 || hi == 0 ? ~0u : 0u;
          u32x4 a4[4];
#pragma unroll
          for (int m = 0; m < 4; ++m)
            a4[m] = ld_b(sx, slot[(jp + 2) % 3] + aof[st] + m * 512);
#pragma unroll
          for (int kd = 0; kd < 3; ++kd) {
            int const oi = jp - kd;  // output plane d0 + oi = p + 1 - kd
            if (oi >= 0 && oi < DB) {
#pragma unroll
              for (int tt = 0; tt < NT; ++tt) {
                u32x4 bt = ld_b(sw, bof + (kd * 9 + 2 * st) * CO * 32 + tt * 512);
                if (st == 4) bt = bt & keep;
#pragma unroll
                for (int m = 0; m < 4; ++m) acc[oi][m][tt] = mfma32(bt, a4[m], acc[oi][m][tt]);
              }
            }
          }
        }
        if (more) {
          __syncthreads();  // every wave is done with plane p
          store_plane(p + 3, nxt);
          __syncthreads();
        }
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < DB; ++j) {
      int const d = d0 + j;
      // plane d + 2 is loaded while plane d is computed, then stored into
      // the slot of plane d - 1
      uint4 nxt[NPK];
      if (j + 1 < DB)
        load_plane(d + 2, c, nxt);
      else if (pre)
        load_chunk(c + 1);
      else if (UPC && c + 1 == CI / 16)
        load_coarse(0);
      __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the compute
      // operands of step st (taps 2 st, 2 st + 1), double-buffered so the
      // LDS reads of the next step overlap this step's MFMAs
      // (the slots pass through an empty asm: their sums with aof, 42 of them,
      // must not be kept over the planes and chunks, which spilled)
      int sl[3] = {slot[(j + 2) % 3], slot[j % 3], slot[(j + 1) % 3]};
#pragma unroll
      for (int q = 0; q < 3; ++q) asm volatile("" : "+s"(sl[q]));
      auto load_ops = [&](int st, Ops &o) {
        int const kd0 = 2 * st / 9, kd1 = 2 * st + 1 < 27 ? (2 * st + 1) / 9 : 2;
        int const s0 = sl[kd0], s1 = sl[kd1];
        int const ab = aof[st] + (kd0 == kd1 ? s0 : hi ? s1 : s0);
#pragma unroll
        for (int m = 0; m < 4; ++m) o.a[m] = ld_b(sx, ab + m * 512);
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) o.b[tt] = ld_b(sw, bof + 2 * st * CO * 32 + tt * 512);
      };
      auto mma_ops = [&](Ops const &o) {
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
          for (int m = 0; m < 4; ++m) acc[j][m][tt] = mfma32(o.b[tt], o.a[m], acc[j][m][tt]);
      };
      Ops opa, opb;
      load_ops(0, opa);
#pragma unroll
      for (int st = 1; st < 14; st += 2) {
        load_ops(st, opb);
        mma_ops(opa);
        if (st + 1 < 14) load_ops(st + 1, opa);
        mma_ops(opb);
      }
      if (j + 1 < DB) {
        __syncthreads();  // every wave is done with plane d - 1
        store_plane(d + 2, nxt);
        __syncthreads();
      }
    }
  }
  coarse_part();
  // Epilogue per plane: each wave writes its row (bias, ReLU applied) into
  // its own LDS rows [voxel][OBS] (lane (i, kq) holds channels t * 16 + 4 kq
  // + r of voxel 16 m + i; padded rows spread the banks), then stores 16-byte
  // pieces of 8 channels, coalesced.
  int const h = h0 + wave;
  uint16_t *const ob = smem + wave * 64 * OBS;
#pragma unroll
  for (int j = 0; j < DB; ++j) {
    int const d = d0 + j;
    __syncthreads();  // the LDS is free (j = 0: done with the operands)
    auto rows = [&](auto relu) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        f32x4 const b = (mode & 1) ? *(f32x4u const *)(bias + t * 16 + 4 * kq)
                                   : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < 4; ++m)
          *(uint2 *)(ob + (16 * m + i) * OBS + t * 16 + 4 * kq) =
              out4<decltype(relu)::value>(acc[j][m][t], b);
      }
    };
    if (mode & 2)
      rows(std::true_type{});
    else
      rows(std::false_type{});
    __syncthreads();
    if (h < H && d < D) {
      int64_t const orow = (((int64_t)n * D + d) * H + h) * W;
      constexpr int C8 = CO / 8;
#pragma unroll
      for (int k = 0; k < (64 * C8 + 63) / 64; ++k) {
        int const e = lane + 64 * k;
        int const v = e / C8, c8 = e - v * C8;
        int const wv = w0 + v;
        if (e < 64 * C8 && wv < W) {
          uint2 const lo = *(uint2 const *)(ob + v * OBS + c8 * 8);
          uint2 const hi = *(uint2 const *)(ob + v * OBS + c8 * 8 + 4);
          uint4 val = make_uint4(lo.x, lo.y, hi.x, hi.y);
          int64_t const o = (orow + wv) * CO + c8 * 8;
          if (mode & 4) {
            uint4 const g = *(uint4 const *)(gate + o);
            uint32_t const gw[4] = {g.x, g.y, g.z, g.w};
            uint32_t vw[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              uint32_t const m0 = bf2f((uint16_t)(gw[q] & 0xffffu)) > 0.f ? 0xffffu : 0u;
              uint32_t const m1 = bf2f((uint16_t)(gw[q] >> 16)) > 0.f ? 0xffff0000u : 0u;
              vw[q] &= m0 | m1;
            }
            val = make_uint4(vw[0], vw[1], vw[2], vw[3]);
          }
          *(uint4 *)(y + o) = val;
        }
      }
    }
    if constexpr (DB % 2 == 0) {
      if (mode & 8) {
        // 2x2x2 max pooling of the output (D, H, W even; d0, h0, w0 even):
        // item (pooled row pr, column pc, 8 channels) scans its voxels in
        // (d, h, w) order with a strict >, as the pooling kernel does; the
        // even plane's partial (one of the bf16 values, so exact) waits in
        // LDS for the odd plane, handled by the same thread
        constexpr int C8 = CO / 8;
        uint16_t *const pm = smem + 4 * 64 * OBS;
        for (int e = tid; e < 2 * 32 * C8; e += UT) {
          int const c8 = e % C8, pc = (e / C8) % 32, pr = e / (C8 * 32);
          float best[8];
          if (j % 2 == 0) {
#pragma unroll
            for (int k = 0; k < 8; ++k) best[k] = -INFINITY;
          } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) best[k] = bf2f(pm[(pr * 32 + pc) * CO + c8 * 8 + k]);
          }
#pragma unroll
          for (int o = 0; o < 4; ++o) {
            uint16_t const *const r =
                smem + (2 * pr + (o >> 1)) * 64 * OBS + (2 * pc + (o & 1)) * OBS + c8 * 8;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              float const f = bf2f(r[k]);
              if (f > best[k]) best[k] = f;
            }
          }
          if (j % 2 == 0) {
#pragma unroll
            for (int k = 0; k < 8; ++k) pm[(pr * 32 + pc) * CO + c8 * 8 + k] = f2bf(best[k]);
          } else {
            int const dp = d / 2, hp = h0 / 2 + pr, wp = w0 / 2 + pc;
            if (d < D && 2 * hp < H && 2 * wp < W) {
              uint32_t q[4];
#pragma unroll
              for (int k = 0; k < 4; ++k)
                q[k] = (uint32_t)f2bf(best[2 * k]) | ((uint32_t)f2bf(best[2 * k + 1]) << 16);
              int64_t const po =
                  ((((int64_t)n * (D / 2) + dp) * (H / 2) + hp) * (W / 2) + wp) * CO + c8 * 8;
              *(uint4 *)(pool + po) = make_uint4(q[0], q[1], q[2], q[3]);
            }
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// 16 -> 16 channels, streaming over the input planes: each input plane is
// staged into LDS once (double-buffered) and each of its A fragments is read
// once and used for the three depth taps, i.e. for the three output planes
// the plane touches (kd = 0, 1, 2 into outputs p + 1, p, p - 1), with the
// weights of all 27 taps in registers. K = 32 pairs two (kh, kw) positions
// of one input plane: step s takes positions 2 s and 2 s + 1 (the tenth
// position, past the ninth, reads the ninth with zero weights). Per 16
// voxels and input plane this reads 5 A fragments from LDS and no B, where
// k_conv3 reads 14 A and 14 B fragments per 16 voxels and output plane.
// Block: CT_H rows x CT_W voxels of DB output planes; without pooling one
// row per wave, with it (POOL) two rows x 32 voxels per wave (wave w: rows
// 2 (w >> 1) + (m >> 1), voxels 32 (w & 1) + 16 (m & 1) + 0..15 of its
// 16-voxel tiles m), so that a lane holds every voxel of its 2 x 2 pooling
// windows (the w pair in one tile, the h pair in tiles m and m + 2).
// Epilogue per output plane: bias and ReLU (mode bits 1, 2), the wave's
// voxels through its own LDS rows as 16-byte coalesced stores; POOL (mode
// bit 8): the 2x2x2 max pooling (k_maxpool's scan order and strict >) in
// registers, the even plane's partial kept for the odd one (D, H, W even,
// DB even).
// grid: (ceil(W / CT_W), ceil(H / CT_H), N * ceil(D / DB)); block 256.
// ---------------------------------------------------------------------------
template <int DB, bool POOL>
__global__ __launch_bounds__(UT, 2) void k_conv3s(uint16_t const *__restrict__ x,
                                               uint16_t const *__restrict__ wt,
                                               float const *__restrict__ bias,
                                               uint16_t *__restrict__ y,
                                               uint16_t *__restrict__ pool, int D, int H, int W,
                                               int mode) {
  static_assert(DB % 2 == 0, "pooling pairs the planes of a block");
  constexpr int PW = CT_W + 2, PH = CT_H + 2;
  constexpr int PLANE = PH * PW * 16;  // bf16 elements of one staged plane
  constexpr int NPI = PH * PW * 2;     // staging items (8 channels) per plane
  constexpr int NPK = (NPI + UT - 1) / UT;
  constexpr int OBS = 16 + 4;               // output row: 16 channels + 4 (bank spread)
  constexpr int ROWS = CT_H * 64 * OBS;     // one output plane's rows
  static_assert(CT_H == 4 && CT_W == 64 && UT == 256, "four waves of 64 voxels");
  __shared__ __align__(16) uint16_t sx[2 * PLANE];
  __shared__ __align__(16) uint16_t so[2 * ROWS];
  int const tid = threadIdx.x;
  int const lane = tid & 63;
  int const wave = tid >> 6;
  int const ndb = (D + DB - 1) / DB;
  int const n = blockIdx.z / ndb;
  int const d0 = (blockIdx.z - n * ndb) * DB;
  int const h0 = blockIdx.y * CT_H;
  int const w0 = blockIdx.x * CT_W;
  // weights as the A operand, voxels as the B (k_conv3): a lane ends with the
  // output channels 4 kq .. + 3 of voxel i of each tile
  int const i = lane & 15;   // output channel (weights), voxel (input, output)
  int const kq = lane >> 4;  // channels 8 (kq & 1) .. + 7 of position 2 s + (kq >> 1)
  uint16_t const *const xn = x + (int64_t)n * D * H * W * 16;
  int64_t const plane = (int64_t)H * W * 16;
  // the weights of every tap: bw[kd][s] = w[kd 9 + 2 s + (kq >> 1)][i][8 (kq & 1) ..]
  u32x4 bw[3][5];
#pragma unroll
  for (int kd = 0; kd < 3; ++kd)
#pragma unroll
    for (int s = 0; s < 5; ++s) {
      int const q = 2 * s + (kq >> 1);
      u32x4 const v = *(u32x4 const *)(wt + ((int64_t)(kd * 9 + (q < 9 ? q : 8)) * 16 + i) * 16 +
                                       8 * (kq & 1));
      unsigned const keep = q < 9 ? ~0u : 0u;
      bw[kd][s] = v & keep;
    }
  // staging items: 32-bit offset within a plane and whether (h, w) lies
  // inside the volume; items past the last repeat it (no branch)
  uint32_t ioff[NPK];
  bool iok[NPK];
#pragma unroll
  for (int k = 0; k < NPK; ++k) {
    int const e0 = tid + k * UT;
    int const e = e0 < NPI ? e0 : NPI - 1;
    int const half = e & 1, r = e >> 1;
    int const pw = r % PW, ph = r / PW;
    int const hh = h0 + ph - 1, ww = w0 + pw - 1;
    iok[k] = hh >= 0 && hh < H && ww >= 0 && ww < W;
    ioff[k] = iok[k] ? (uint32_t)(hh * W + ww) * 16u + (uint32_t)(half * 8) : (uint32_t)(half * 8);
  }
  auto load_plane = [&](int dd, uint4 (&v)[NPK]) {
    bool const okd = dd >= 0 && dd < D;
    uint16_t const *const src = xn + (okd ? dd : 0) * plane;
#pragma unroll
    for (int k = 0; k < NPK; ++k) {
      uint32_t const msk = (okd && iok[k]) ? ~0u : 0u;
      uint4 const t = *(uint4 const *)(src + ioff[k]);
      v[k] = make_uint4(t.x & msk, t.y & msk, t.z & msk, t.w & msk);
    }
  };
  auto store_plane = [&](uint16_t *dst, uint4 const (&v)[NPK]) {
#pragma unroll
    for (int k = 0; k < NPK; ++k) {
      int const e0 = tid + k * UT;
      int const e = e0 < NPI ? e0 : NPI - 1;
      st_h(dst, e >> 1, e & 1, v[k]);  // past the end: the last item again
    }
  };
  f32x4 acc[DB][4];
#pragma unroll
  for (int j = 0; j < DB; ++j)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  // row and first voxel (within the block) of the wave's tile m
  auto trow = [&](int m) { return POOL ? 2 * (wave >> 1) + (m >> 1) : wave; };
  auto tcol = [&](int m) { return POOL ? 32 * (wave & 1) + 16 * (m & 1) : 16 * m; };
  // loaded once: a load in the loop would be issued after the next plane's
  // prefetch, and waiting for it would wait for the prefetch too
  f32x4 const b =
      (mode & 1) ? *(f32x4u const *)(bias + 4 * kq) : f32x4{0.f, 0.f, 0.f, 0.f};
  // LDS byte offsets of the lane's voxels in a plane, per step and (POOL)
  // tile row: the loop adds constants only
  int aof[POOL ? 2 : 1][5];
#pragma unroll
  for (int q = 0; q < (POOL ? 2 : 1); ++q)
#pragma unroll
    for (int s = 0; s < 5; ++s) {
      int const u = 2 * s + (kq >> 1), t = u < 9 ? u : 8;
      aof[q][s] = off_h((trow(2 * q) + t / 3) * PW + tcol(0) + i + t % 3, kq & 1);
    }
  // POOL: the even plane's pooling partials of this lane's two voxel rows'
  // channels, per tile column mc (bf16 values, so exact)
  float pp[2][4];
#pragma unroll
  for (int q = 0; q < 8; ++q) pp[q >> 2][q & 3] = -INFINITY;
  // output plane oi (d0 + oi): bias, ReLU, into the wave's rows of buffer
  // oi & 1, then stored by the wave itself; POOL: its pooling
  auto epilogue = [&](int oi) {
    int const d = d0 + oi;
    uint16_t *const ob = so + (oi & 1) * ROWS + wave * 64 * OBS;
    uint2 pk[4];
    if (mode & 2) {
#pragma unroll
      for (int m = 0; m < 4; ++m) pk[m] = out4<true>(acc[oi][m], b);
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) pk[m] = out4<false>(acc[oi][m], b);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) *(uint2 *)(ob + (16 * m + i) * OBS + 4 * kq) = pk[m];
    __builtin_amdgcn_wave_barrier();
    if (d < D) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        int const e = lane + 64 * k;  // (voxel of the wave, 8-channel half)
        int const v = e >> 1, c8 = e & 1;
        int const hh = h0 + trow(v >> 4), ww = w0 + tcol(v >> 4) + (v & 15);
        if (hh < H && ww < W) {
          uint2 const lo = *(uint2 const *)(ob + v * OBS + c8 * 8);
          uint2 const hi = *(uint2 const *)(ob + v * OBS + c8 * 8 + 4);
          *(uint4 *)(y + ((((int64_t)n * D + d) * H + hh) * W + ww) * 16 + c8 * 8) =
              make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
      }
    }
    if constexpr (POOL) {
      // pooling window of tile column mc: voxel i (and lane i + 1's, for even
      // i) of tiles mc, mc + 2, scanned in (h, w) order with a strict >, after
      // the even plane's
      bool const odd = oi & 1;
#pragma unroll
      for (int mc = 0; mc < 2; ++mc) {
        uint2 const own[2] = {pk[mc], pk[mc + 2]};
        uint2 nb[2];
#pragma unroll
        for (int q = 0; q < 2; ++q)
          nb[q] = make_uint2(__shfl_xor(own[q].x, 1, 64), __shfl_xor(own[q].y, 1, 64));
        uint32_t pq[2] = {0, 0};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          auto ch = [&](uint2 v) {
            uint32_t const u = r < 2 ? v.x : v.y;
            return __uint_as_float(r & 1 ? u & 0xffff0000u : u << 16);
          };
          float best = odd ? pp[mc][r] : -INFINITY;
#pragma unroll
          for (int o = 0; o < 4; ++o) {
            float const f = ch(o & 1 ? nb[o >> 1] : own[o >> 1]);
            if (f > best) best = f;
          }
          pp[mc][r] = best;
          pq[r >> 1] |= (__float_as_uint(best) >> 16) << (16 * (r & 1));  // a bf16 value
        }
        if (odd && !(i & 1)) {
          int const dp = d / 2, hp = h0 / 2 + (wave >> 1);
          int const wp = w0 / 2 + 16 * (wave & 1) + 8 * mc + i / 2;
          if (d < D && 2 * hp < H && 2 * wp < W)
            *(uint2 *)(pool + ((((int64_t)n * (D / 2) + dp) * (H / 2) + hp) * (W / 2) + wp) * 16 +
                       4 * kq) = make_uint2(pq[0], pq[1]);
        }
      }
    }
  };
  // AH2: two planes in flight per block (nxt, nx2), since the loads a CU
  // keeps in flight set this layer's HBM rate (with pooling the registers
  // would spill: one plane)
  constexpr bool AH2 = !POOL;
  uint4 nxt[NPK], nx2[AH2 ? NPK : 1];
  {
    uint4 v0[NPK];
    load_plane(d0 - 1, v0);
    load_plane(d0, nxt);
    if constexpr (AH2) load_plane(d0 + 1, nx2);
    store_plane(sx, v0);
  }
  __syncthreads();
  // input plane p = d0 - 1 + j is in buffer j & 1; nxt holds plane p + 1,
  // stored into the other buffer (free: every wave passed the barrier after
  // reading it); then (AH2) nx2's plane p + 2 moves to nxt while plane p + 3
  // is loaded into nx2, or plane p + 2 is loaded into nxt
#pragma unroll
  for (int j = 0; j < DB + 2; ++j) {
    uint16_t const *const cur = sx + (j & 1) * PLANE;
    if (j + 1 < DB + 2) {
      store_plane(sx + ((j + 1) & 1) * PLANE, nxt);
      if constexpr (AH2) {
#pragma unroll
        for (int k = 0; k < NPK; ++k) nxt[k] = nx2[k];
        if (j + 3 < DB + 2) load_plane(d0 + 2 + j, nx2);
      } else if (j + 2 < DB + 2) {
        load_plane(d0 + 1 + j, nxt);
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the compute
    }
#pragma unroll
    for (int s = 0; s < 5; ++s) {
      u32x4 a[4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
        a[m] = ld_b(cur, (POOL ? aof[m >> 1][s] + (m & 1) * 512 : aof[0][s] + m * 512));
#pragma unroll
      for (int kd = 0; kd < 3; ++kd) {
        int const oi = j - kd;  // output plane d0 + oi = p + 1 - kd
        if (oi >= 0 && oi < DB) {
#pragma unroll
          for (int m = 0; m < 4; ++m) acc[oi][m] = mfma32(bw[kd][s], a[m], acc[oi][m]);
        }
      }
    }
    if (j >= 2) epilogue(j - 2);
    __syncthreads();
  }
}

// Combined taps of the first CU input channels of wt ([27][CO][CI]):
// wcu[((pd 2 + ph) 4 + a 2 + b) 3 + kw][co][cu] = bf16(sum over the d taps kd of
// (pd, a) and the h taps kh of (ph, b) of wt[(kd * 3 + kh) * 3 + kw][co][cu]),
// summed in fp32 in tap order. Taps of parity p and pair index a: p = 0:
// {0}, {1, 2}; p = 1: {0, 1}, {2}.
__global__ __launch_bounds__(UT) void k_up_weights(uint16_t const *__restrict__ wt,
                                                   uint16_t *__restrict__ wcu, int CI, int CO,
                                                   int CU) {
  int const n = 48 * CO * CU;
  for (int e = blockIdx.x * UT + threadIdx.x; e < n; e += gridDim.x * UT) {
    int const cu = e % CU;
    int const co = (e / CU) % CO;
    int const tap = e / (CU * CO);
    int const kw = tap % 3, ab = (tap / 3) % 4, pp = tap / 12;
    int const pd = pp >> 1, ph = pp & 1, a = ab >> 1, b = ab & 1;
    int const dlo = (pd == 0) ? (a == 0 ? 0 : 1) : (a == 0 ? 0 : 2);
    int const dhi = (pd == 0) ? (a == 0 ? 0 : 2) : (a == 0 ? 1 : 2);
    int const hlo = (ph == 0) ? (b == 0 ? 0 : 1) : (b == 0 ? 0 : 2);
    int const hhi = (ph == 0) ? (b == 0 ? 0 : 2) : (b == 0 ? 1 : 2);
    float acc = 0.f;
    for (int kd = dlo; kd <= dhi; ++kd)
      for (int kh = hlo; kh <= hhi; ++kh)
        acc += bf2f(wt[((int64_t)((kd * 3 + kh) * 3 + kw) * CO + co) * CI + cu]);
    wcu[e] = f2bf(acc);
  }
}

// ---------------------------------------------------------------------------
// First layer: one live input channel (the field), so the taps are the GEMM's
// K: D[voxel][co] = sum_tap bf16(field[voxel + tap] * scale) w[tap][co][0],
// K = 27 taps padded to 32 (one K = 32 step) instead of 27 steps of 16
// channels. Block: CT_H rows x CT_W voxels of FDB consecutive d planes, a
// ring of three bf16 planes of the field in LDS; output as in k_conv3
// (bias, ReLU, 16-byte stores through per-wave LDS rows).
// grid: (ceil(W / CT_W), ceil(H / CT_H), N * ceil(D / FDB)); block 256.
// ---------------------------------------------------------------------------
#define FDB 16
__global__ __launch_bounds__(UT) void k_conv_first(float const *__restrict__ src,
                                                   uint16_t const *__restrict__ wt, int wci,
                                                   float const *__restrict__ bias,
                                                   uint16_t *__restrict__ y, int D, int H,
                                                   int W, float scale) {
  constexpr int PW = CT_W + 2, PH = CT_H + 2, PLANE = PH * PW;
  constexpr int OBS = 20;
  __shared__ __align__(16) uint16_t sx[3 * PLANE];
  __shared__ __align__(16) uint16_t ob[4 * 64 * OBS];
  int const tid = threadIdx.x;
  int const lane = tid & 63, wave = tid >> 6;
  int const i = lane & 15, kq = lane >> 4;
  int const ndb = (D + FDB - 1) / FDB;
  int const n = blockIdx.z / ndb;
  int const d0 = (blockIdx.z - n * ndb) * FDB;
  int const h0 = blockIdx.y * CT_H, w0 = blockIdx.x * CT_W;
  float const *const fn = src + (int64_t)n * D * H * W;
  // B: taps 8 kq + e of output channel i (zero past tap 26): K = 32
  unsigned bh[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    int const t = 8 * kq + e;
    bh[e] = t < 27 ? (unsigned)wt[((int64_t)t * 16 + i) * wci] : 0u;
  }
  u32x4 const bw = {bh[0] | bh[1] << 16, bh[2] | bh[3] << 16, bh[4] | bh[5] << 16,
                    bh[6] | bh[7] << 16};
  // LDS offsets of this lane's A taps relative to its voxel (slot, row, col)
  int toff[8], tkd[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    int const t = 8 * kq + e;
    int const tt = t < 27 ? t : 13;  // padded taps read the centre (weight 0)
    tkd[e] = tt / 9;
    toff[e] = ((tt / 3) % 3) * PW + tt % 3;
  }
  // a plane's field values: raw loads at clamped offsets, converted and
  // zeroed outside the volume when stored, so that the next plane's loads
  // stay in flight while the current one is computed
  constexpr int NPK = (PLANE + UT - 1) / UT;
  int foff[NPK];
  bool fok[NPK];
#pragma unroll
  for (int k = 0; k < NPK; ++k) {
    int const e = min(tid + k * UT, PLANE - 1);
    int const ph = e / PW, pw = e - ph * PW;
    int const hh = h0 + ph - 1, ww = w0 + pw - 1;
    fok[k] = hh >= 0 && hh < H && ww >= 0 && ww < W;
    foff[k] = fok[k] ? hh * W + ww : 0;
  }
  auto load_plane = [&](int dd, float (&v)[NPK]) {
    float const *const src = fn + (int64_t)(dd >= 0 && dd < D ? dd : 0) * H * W;
#pragma unroll
    for (int k = 0; k < NPK; ++k) v[k] = src[foff[k]];
  };
  auto store_plane = [&](int dd, float const (&v)[NPK]) {
    uint16_t *const dst = sx + ((dd + 3) % 3) * PLANE;
    bool const okd = dd >= 0 && dd < D;
#pragma unroll
    for (int k = 0; k < NPK; ++k) {
      int const e = tid + k * UT;
      if (e < PLANE) dst[e] = (okd && fok[k]) ? f2bf(v[k] * scale) : (uint16_t)0;
    }
  };
  float const bsel = bias[i];
  // two planes in flight: nv holds plane d + 1 (stored at the top of the
  // iteration), nv2 plane d + 2 (moved to nv while plane d + 3 is loaded)
  float nv[NPK], nv2[NPK];
  load_plane(d0 - 1, nv);
  store_plane(d0 - 1, nv);
  load_plane(d0, nv);
  store_plane(d0, nv);
  load_plane(d0 + 1, nv);
  load_plane(d0 + 2, nv2);
  int const h = h0 + wave;
  uint16_t *const obw = ob + wave * 64 * OBS;
  for (int j = 0; j < FDB; ++j) {
    int const d = d0 + j;
    store_plane(d + 1, nv);
#pragma unroll
    for (int k = 0; k < NPK; ++k) nv[k] = nv2[k];
    if (j + 2 < FDB) load_plane(d + 3, nv2);
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the compute
    __syncthreads();
    f32x4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      int const vb = wave * PW + 16 * m + i;  // the voxel's (row, col) in a plane
      unsigned ah[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        ah[e] = sx[((d + tkd[e] - 1 + 3) % 3) * PLANE + vb + toff[e]];
      u32x4 const a = {ah[0] | ah[1] << 16, ah[2] | ah[3] << 16, ah[4] | ah[5] << 16,
                       ah[6] | ah[7] << 16};
      acc[m] = mfma32(a, bw, acc[m]);
    }
    // D: lane holds voxels 16 m + 4 kq + r of channel i
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        obw[(16 * m + 4 * kq + r) * OBS + i] = f2bf(fmaxf(acc[m][r] + bsel, 0.f));
    __syncthreads();  // the output rows are complete; the ring slot of d - 1 is free
    if (h < H && d < D) {
      int64_t const orow = (((int64_t)n * D + d) * H + h) * W;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        int const e = lane + 64 * k;  // (voxel, 8-channel half)
        int const v = e >> 1, c8 = e & 1;
        if (w0 + v < W) {
          uint2 const lo = *(uint2 const *)(obw + v * OBS + c8 * 8);
          uint2 const hi = *(uint2 const *)(obw + v * OBS + c8 * 8 + 4);
          *(uint4 *)(y + (orow + w0 + v) * 16 + c8 * 8) = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Head: output channel 0 of a 16 -> 16 convolution, in fp32, plus the field:
// out[v] = base[v] + s (b0 + sum_tap sum_ci x[v + tap][ci] w[tap][0][ci]).
// For an output plane d, F[u][(kh, kw)] = sum_kd sum_ci x_{d+kd-1}[u][ci]
// w[(kd, kh, kw)][0][ci] over every staged voxel u (halo included) is a GEMM
// with M = voxels, K = (kd, ci) = 48 and N = 9 taps (padded to 16): two
// K = 32 MFMAs per 16 voxels (planes d - 1 and d, then plane d + 1 with the
// second half's weights zero). Then out[v] gathers F[v + (kh - 1, kw - 1)]
// [(kh, kw)], 9 terms. Block: CT_H rows x CT_W voxels of HDB consecutive d
// planes, the input planes in a ring of three (16-byte halves swizzled as in
// k_conv3), the next plane loaded while the current one is computed.
// grid: (ceil(W / CT_W), ceil(H / CT_H), N * ceil(D / HDB)); block 256.
// ---------------------------------------------------------------------------
#define HDB 16
__global__ __launch_bounds__(UT) void k_conv_head(uint16_t const *__restrict__ x,
                                                  uint16_t const *__restrict__ wt, int wco,
                                                  float const *__restrict__ bias,
                                                  float const *__restrict__ base,
                                                  float *__restrict__ dst, int D, int H, int W,
                                                  float unscale) {
  constexpr int PW = CT_W + 2, PH = CT_H + 2;
  constexpr int NV = PH * PW;           // staged voxels per plane (396)
  constexpr int NVT = (NV + 15) / 16;   // 16-voxel tiles (25)
  constexpr int PLANE = NV * 16;        // bf16 elements per staged plane
  constexpr int NPI = NV * 2;           // staging items of 8 channels
  constexpr int NPK = (NPI + UT - 1) / UT;
  // F tap-major, one row of NVP >= 16 NVT floats per tap: a lane's four
  // consecutive voxels of one tap are one 16-byte write, and NVP = 20 mod 32
  // spreads the eight lanes of a write cycle over distinct bank groups
  constexpr int NVP = 404;
  static_assert(NVP >= NVT * 16 && NVP % 32 == 20, "F rows");
  __shared__ __align__(16) uint16_t sx[3 * PLANE];
  __shared__ __align__(16) float se[9 * NVP];
  int const tid = threadIdx.x;
  int const lane = tid & 63, wave = tid >> 6;
  int const i = lane & 15, kq = lane >> 4;
  int const ndb = (D + HDB - 1) / HDB;
  int const n = blockIdx.z / ndb;
  int const d0 = (blockIdx.z - n * ndb) * HDB;
  int const h0 = blockIdx.y * CT_H, w0 = blockIdx.x * CT_W;
  uint16_t const *const xn = x + (int64_t)n * D * H * W * 16;
  int64_t const plane = (int64_t)H * W * 16;
  // B: lane (tap i, k group kq) holds input channels 8 (kq & 1) .. + 7 of
  // depth tap kd = kq >> 1 (bw0) and kd = 2 for kq < 2, zero for kq >= 2
  // (bw1), of output channel 0; taps i >= 9 zero
  u32x4 bw0, bw1;
  {
    unsigned h0w[8], h1w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int const ci = 8 * (kq & 1) + e;
      h0w[e] = i < 9 ? (unsigned)wt[((int64_t)((kq >> 1) * 9 + i) * wco) * 16 + ci] : 0u;
      h1w[e] = (i < 9 && kq < 2) ? (unsigned)wt[((int64_t)(18 + i) * wco) * 16 + ci] : 0u;
    }
    bw0 = u32x4{h0w[0] | h0w[1] << 16, h0w[2] | h0w[3] << 16, h0w[4] | h0w[5] << 16,
                h0w[6] | h0w[7] << 16};
    bw1 = u32x4{h1w[0] | h1w[1] << 16, h1w[2] | h1w[3] << 16, h1w[4] | h1w[5] << 16,
                h1w[6] | h1w[7] << 16};
  }
  uint32_t ioff[NPK];
  bool iok[NPK];
#pragma unroll
  for (int k = 0; k < NPK; ++k) {
    int const e0 = tid + k * UT;
    int const e = e0 < NPI ? e0 : NPI - 1;
    int const half = e & 1, r = e >> 1;
    int const pw = r % PW, ph = r / PW;
    int const hh = h0 + ph - 1, ww = w0 + pw - 1;
    iok[k] = hh >= 0 && hh < H && ww >= 0 && ww < W;
    ioff[k] = iok[k] ? (uint32_t)(hh * W + ww) * 16u + (uint32_t)(half * 8) : (uint32_t)(half * 8);
  }
  // the loads are raw (clamped addresses); the halo and out-of-range planes
  // are zeroed when the plane is stored, so that a prefetch stays in flight
  // until then
  auto load_plane = [&](int dd, uint4 (&v)[NPK]) {
    bool const okd = dd >= 0 && dd < D;
    uint16_t const *const src = xn + (okd ? dd : 0) * plane;
#pragma unroll
    for (int k = 0; k < NPK; ++k) v[k] = *(uint4 const *)(src + ioff[k]);
  };
  auto store_plane = [&](int dd, uint4 const (&v)[NPK]) {
    bool const okd = dd >= 0 && dd < D;
    uint16_t *const dstp = sx + ((dd + 3) % 3) * PLANE;
#pragma unroll
    for (int k = 0; k < NPK; ++k) {
      int const e0 = tid + k * UT;
      int const e = e0 < NPI ? e0 : NPI - 1;
      uint32_t const msk = (okd && iok[k]) ? ~0u : 0u;
      st_h(dstp, e >> 1, e & 1, make_uint4(v[k].x & msk, v[k].y & msk, v[k].z & msk, v[k].w & msk));
    }
  };
  {
    uint4 v0[NPK], v1[NPK], v2[NPK];
    load_plane(d0 - 1, v0);
    load_plane(d0, v1);
    load_plane(d0 + 1, v2);
    store_plane(d0 - 1, v0);
    store_plane(d0, v1);
    store_plane(d0 + 1, v2);
  }
  int const row = tid >> 6, col = tid & 63;
  float const b0 = bias[0];
  constexpr int TPW = (NVT + UT / 64 - 1) / (UT / 64);  // tiles per wave
  for (int j = 0; j < HDB; ++j) {
    int const d = d0 + j;
    int const h = h0 + row, w = w0 + col;
    bool const live = h < H && w < W && d < D;
    int64_t const v = (((int64_t)n * D + (live ? d : 0)) * H + (live ? h : 0)) * W + (live ? w : 0);
    // the field value is loaded before the prefetch, so that waiting for
    // it does not wait for the prefetch
    float const bv = base ? base[v] : 0.f;
    uint4 nxt[NPK];
    if (j + 1 < HDB) load_plane(d + 2, nxt);
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the compute
    __syncthreads();  // the ring holds planes d - 1, d, d + 1; F is free
    {
      // lanes kq < 2 read plane d - 1 (first MFMA) and d + 1 (second), lanes
      // kq >= 2 plane d (first) and d + 1 again (second: zero weights)
      uint16_t const *const p1 = sx + ((kq < 2 ? d + 2 : d) % 3) * PLANE;
      uint16_t const *const p2 = sx + ((d + 1) % 3) * PLANE;
      u32x4 a1[TPW], a2[TPW];
#pragma unroll
      for (int q = 0; q < TPW; ++q) {
        int const u = (wave + q * (UT / 64)) * 16 + i;
        a1[q] = ld_h(p1, u < NV ? u : NV - 1, kq & 1);
        a2[q] = ld_h(p2, u < NV ? u : NV - 1, kq & 1);
      }
#pragma unroll
      for (int q = 0; q < TPW; ++q) {
        int const t = wave + q * (UT / 64);
        if (t < NVT) {
          f32x4 e = {0.f, 0.f, 0.f, 0.f};
          e = mfma32(a1[q], bw0, e);
          e = mfma32(a2[q], bw1, e);
          // D: lane holds voxels 16 t + 4 kq + r of tap i
          if (i < 9) *(f32x4 *)(se + i * NVP + t * 16 + 4 * kq) = e;
        }
      }
    }
    __syncthreads();  // F is complete; every wave is done with the ring
    if (j + 1 < HDB) store_plane(d + 2, nxt);  // into the slot of plane d - 1
    float acc = 0.f;
#pragma unroll
    for (int kh = 0; kh < 3; ++kh)
#pragma unroll
      for (int kw = 0; kw < 3; ++kw)
        acc += se[(kh * 3 + kw) * NVP + (row + kh) * PW + col + kw];
    if (live) {
      float const o = (acc + b0) * unscale;
      dst[v] = base ? bv + o : o;
    }
  }
}

// wt_t[tap][ci][co] = wt[26 - tap][co][ci]: the weights of the input
// gradient (a convolution of dy with the flipped kernel, CO -> CI channels)
__global__ void k_flip_weights(uint16_t const *__restrict__ wt, uint16_t *__restrict__ wtt,
                               int CI, int CO) {
  int const idx = blockIdx.x * blockDim.x + threadIdx.x;
  int const total = 27 * CI * CO;
  if (idx >= total) return;
  int const tap = idx / (CI * CO);
  int const r = idx - tap * CI * CO;
  int const ci = r / CO;
  int const co = r - ci * CO;
  wtt[idx] = wt[((int64_t)(26 - tap) * CO + co) * CI + ci];
}

// ---------------------------------------------------------------------------
// Weight and bias gradients: dW[tap][co][ci] = sum_v dy[v][co] x[v + tap][ci],
// db[co] = sum_v dy[v][co]
// ---------------------------------------------------------------------------
// A GEMM over voxels (K) on the matrix cores, one 16 x 16 tile pair of
// (output, input) channels per block: per tap A[co][v] = dy and
// B[v][ci] = the shifted input, K = 32 voxels along w per instruction. Rows
// sit in LDS as in memory, [voxel][16 channels], and both operands come
// through the transposing LDS read, so a kw shift is a row offset and
// nothing is transposed when staged. A block owns a 64-voxel w chunk of RB
// consecutive (n, d, h) rows and one kd; its two waves take a 32-voxel half
// each and walk the input rows with the three dy rows (kh) that meet one in
// registers: one new row of each per step, so a step's nine matrix-core
// instructions need four operand reads. The rows of the next two steps are in flight during the current one
// (two register sets, two LDS stages, one barrier per step). A row chunk's
// tile pairs and kd are neighbours on one XCD: they read the same rows, and
// 32 of the 2 CI bytes of a voxel each (pairs apart: 715 us for 48 -> 16
// channels). The sums
// keep one fixed order: a half's rows in turn, the two halves, then the
// blocks (k_reduce_parts). The partial sums go to part[block][27][CO][CI],
// the bias's to bpart[block][CO].
//
// Bound by its loads (dy and x three times). 11 launches of a training step
// on 16 x 32 x 32 x 256: 4.65 ms when rows were staged transposed, once per
// (kh, kw), for 18 instructions a row; 2.64 with the rows as they are and six
// waves a block (all kd), 2.06 so. Input rows against nine dy rows, four d to
// a block, read less and took 1.1 ms, but sum in another order: enough to
// change the second step of Adam in the fifth digit.
#define WG_T 128
// LDS row of voxel v: 32 bytes, 128 more per 8 voxels (the four row groups of
// an operand read then fall in distinct banks)
#define WG_ROW(v) ((v) * 32 + ((v) >> 3) * 128)
#define WG_DY WG_ROW(64)                     // bytes of a stage's dy row
#define WG_X (WG_ROW(65) + 32)               // and of one input row (w0 - 1 .. w0 + 64)
#define WG_STAGE (WG_DY + (WG_X + 127) / 128 * 128)

typedef short s16x4 __attribute__((ext_vector_type(4)));
// 8 voxels of one channel (lane: channel l % 16, voxels 8 (l / 16) + e): two
// transposing reads of 4 rows of 16 channels, at lo and hi
__device__ __forceinline__ u32x4 ld_tr(unsigned char *lo, unsigned char *hi) {
  typedef s16x4 __attribute__((address_space(3))) * lds4;
  s16x4 const a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(s16x4 *)lo);
  s16x4 const b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(s16x4 *)hi);
  uint2 const l = __builtin_bit_cast(uint2, a), h = __builtin_bit_cast(uint2, b);
  return u32x4{l.x, l.y, h.x, h.y};
}

__global__ __launch_bounds__(WG_T, 4) void k_conv3_wgrad(
    uint16_t const *__restrict__ x, uint16_t const *__restrict__ dy, float *__restrict__ part,
    float *__restrict__ bpart, int D, int H, int W, int CI, int CO, int64_t rows, int RB) {
  constexpr int RED = 9 * 256 * 4;
  __shared__ __align__(16) unsigned char lds[2 * WG_STAGE > RED ? 2 * WG_STAGE : RED];
  int const tid = threadIdx.x, lane = tid & 63;
  int const i = lane & 15, kq = lane >> 4;
  int const cs = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (row chunk, input tile, output tile, kd), kd fastest
  int const nct = CO / 16, nsub = 3 * nct * (CI / 16);
  int const id = xcd_chunk(blockIdx.x, gridDim.x);
  int const blk = id / nsub, sub = id - blk * nsub;
  int const kd = sub % 3, ct = sub / 3 % nct, it = sub / 3 / nct;
  int const nwc = (W + 63) / 64;
  int const w0 = (blk % nwc) * 64;
  int64_t const r0 = (int64_t)(blk / nwc) * RB;
  int64_t const r1 = r0 + RB < rows ? r0 + RB : rows;
  // bias sums: channel tid % 16, voxels [vpp p, vpp (p + 1)), p = tid / 16 (+ 8)
  int const npart = 256 / CO, vpp = 64 / npart, pt = tid >> 4;
  bool const do_bias = bpart != nullptr && it == 0 && kd == 1;
  float bsum[2] = {0.f, 0.f};
  f32x4 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the thread's 16-byte items of a stage (voxel, half of its 16 channels):
  // one of the dy row and one of the input row per 64 threads and half, and
  // the input row's two last voxels
  int const v = tid >> 1, half = (tid & 1) * 16;
  int const c8 = (tid & 1) * 8;
  bool const dylive = w0 + v < W, more = tid < 4 && w0 + 63 + v < W;
  bool const xlive = w0 - 1 + v >= 0 && w0 - 1 + v < W;
  int const dyat = WG_ROW(v) + half, xat = WG_DY + dyat, mat = WG_DY + WG_ROW(64 + v) + half;
  // the lane's operand rows: of dy, and of the input row by kw
  int const rl = cs * 32 + 8 * kq + (i >> 2), col = (i & 3) * 8;
  int const alo = col + WG_ROW(rl), ahi = col + WG_ROW(rl + 4);
  int blo[3], bhi[3];
#pragma unroll
  for (int kw = 0; kw < 3; ++kw) {
    blo[kw] = col + WG_DY + WG_ROW(rl + kw);
    bhi[kw] = col + WG_DY + WG_ROW(rl + 4 + kw);
  }
  int buf = 0;
  // runs of rows of one (n, d)
  for (int64_t ra = r0; ra < r1;) {
    int const h0 = (int)(ra % H);
    int64_t const nd = ra / H;
    int const d = (int)(nd % D), dd = d + kd - 1;
    int const h1 = (int)(r1 - ra < H - h0 ? h0 + (r1 - ra) : H);
    ra += h1 - h0;
    bool const plane = dd >= 0 && dd < D;
    // step h = h0 - 1 .. h1: the input row h and the dy row h + 1. Loads are
    // unconditional (a row outside the run or the volume reads the tensor's
    // first voxel and is zeroed).
    uint16_t const *const py = dy + (nd * H * W + w0 + v) * CO + ct * 16 + c8;
    uint16_t const *const px =
        x + ((nd + (kd - 1)) * H * W + (w0 - 1 + v)) * (int64_t)CI + it * 16 + c8;
    struct Rows {
      uint4 y, x, m;
    };
    auto fetch = [&](int h) {
      Rows r;
      bool const oy = dylive && h + 1 < h1, ox = plane && h >= 0 && h < H;
      r.y = *(uint4 const *)(oy ? py + (int64_t)(h + 1) * W * CO : dy);
      r.x = *(uint4 const *)(ox && xlive ? px + (int64_t)h * W * CI : x);
      r.m = make_uint4(0, 0, 0, 0);
      if (tid < 4) r.m = *(uint4 const *)(ox && more ? px + ((int64_t)h * W + 64) * CI : x);
      if (!oy) r.y = make_uint4(0, 0, 0, 0);
      if (!(ox && xlive)) r.x = make_uint4(0, 0, 0, 0);
      if (!(ox && more)) r.m = make_uint4(0, 0, 0, 0);
      return r;
    };
    u32x4 a[3] = {};  // dy rows h + 1 - kh
    auto step = [&](int h, Rows &r) {
      unsigned char *const st = lds + buf * WG_STAGE;
      buf ^= 1;
      *(uint4 *)(st + dyat) = r.y;
      *(uint4 *)(st + xat) = r.x;
      if (tid < 4) *(uint4 *)(st + mat) = r.m;
      __syncthreads();
      if (h + 2 <= h1) r = fetch(h + 2);
      a[2] = a[1];
      a[1] = a[0];
      a[0] = ld_tr(st + alo, st + ahi);
      u32x4 b[3];
#pragma unroll
      for (int kw = 0; kw < 3; ++kw) b[kw] = ld_tr(st + blo[kw], st + bhi[kw]);
      if (do_bias && h + 1 < h1) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          int const p = pt + 8 * u;
          if (p >= npart) continue;
          uint16_t const *const q = (uint16_t const *)st + (tid & 15);
          for (int k = p * vpp; k < (p + 1) * vpp; k += 4) {
            uint16_t const *const z = q + WG_ROW(k) / 2;  // 4 voxels of one group of 8
            bsum[u] += (bf2f(z[0]) + bf2f(z[16])) + (bf2f(z[32]) + bf2f(z[48]));
          }
        }
      }
#pragma unroll
      for (int kh = 0; kh < 3; ++kh) {
        if (h + 1 - kh < h0 || h + 1 - kh >= h1) continue;
#pragma unroll
        for (int kw = 0; kw < 3; ++kw) acc[kh * 3 + kw] = mfma32(a[kh], b[kw], acc[kh * 3 + kw]);
      }
    };
    Rows p0 = fetch(h0 - 1), p1 = fetch(h0);
    for (int h = h0 - 1; h <= h1; h += 2) {
      step(h, p0);
      if (h + 1 <= h1) step(h + 1, p1);
    }
  }
  float *const red = (float *)lds;
  if (do_bias) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (pt + 8 * u < npart) red[tid + 128 * u] = bsum[u];
    __syncthreads();
    if (tid < 16) {
      float s = 0.f;
      for (int q = 0; q < npart; ++q) s += red[q * 16 + tid];
      bpart[(int64_t)blk * CO + ct * 16 + tid] = s;
    }
  }
  // the two halves, then one partial per block
  __syncthreads();
  if (cs == 1) {
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) red[t * 256 + q * 64 + lane] = acc[t][q];
  }
  __syncthreads();
  if (cs == 0) {
    float *const out = part + (int64_t)blk * 27 * CO * CI;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        out[((int64_t)(kd * 9 + t) * CO + ct * 16 + 4 * kq + q) * CI + it * 16 + i] =
            acc[t][q] + red[t * 256 + q * 64 + lane];
  }
}

// The blocks' partial sums in a fixed order: groups of RED_PER blocks, each in
// turn, then the groups in turn. dw: [len] from part [nslab][len]; blocks
// beyond it: db [co] from bpart [nslab][co]. A block takes 16 outputs, 16
// groups at a time: one launch per layer instead of four (11 layers of a step:
// 0.35 ms -> 0.19).
#define RED_PER 32
__global__ __launch_bounds__(UT) void k_reduce_parts(float const *__restrict__ part,
                                                     float *__restrict__ dw, int nslab, int len,
                                                     float const *__restrict__ bpart,
                                                     float *__restrict__ db, int co) {
  __shared__ float sum[16][17];
  int const wblk = (len + 15) / 16;
  bool const bias = (int)blockIdx.x >= wblk;
  int const o = ((int)blockIdx.x - (bias ? wblk : 0)) * 16 + (threadIdx.x & 15);
  int const n = bias ? co : len, slot = threadIdx.x >> 4;
  float const *const src = (bias ? bpart : part) + min(o, n - 1);
  int const ng = (nslab + RED_PER - 1) / RED_PER;
  float total = 0.f;
  for (int g0 = 0; g0 < ng; g0 += 16) {
    int const s0 = (g0 + slot) * RED_PER, s1 = min(s0 + RED_PER, nslab);
    float s = 0.f;
#pragma unroll 8
    for (int k = s0; k < s1; ++k) s += src[(int64_t)k * n];
    sum[slot][threadIdx.x & 15] = s;
    __syncthreads();
    if (slot == 0)
      for (int g = 0; g < min(16, ng - g0); ++g) total += sum[g][threadIdx.x];
    __syncthreads();
  }
  if (slot == 0 && o < n) (bias ? db : dw)[o] = total;
}

// ---------------------------------------------------------------------------
// Pooling, upsampling, concatenation, loss, optimizer
// ---------------------------------------------------------------------------
// Elementwise kernels move 8 channels (16 bytes) per thread; channel counts
// and offsets are multiples of 8 (checked on the host).
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint8_t u8x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ u16x8 ld8(uint16_t const *p) { return *(u16x8 const *)p; }
__device__ __forceinline__ void st8(uint16_t *p, u16x8 v) { *(u16x8 *)p = v; }
typedef uint16_t u16x8u __attribute__((ext_vector_type(8), aligned(2)));

// The training pass's resampling kernels: a thread per 16-byte item (n, d, h,
// w, 8 channels) of their output, its indices by multiplication with the
// sizes' reciprocals where there are fewer than 2^31 items. Pooling and its
// gradient on 64 channels, us: 64-bit divisions per item 58 and 93 at 64 x 64 x
// 512, 20 and 31 at 2 x 2 x 2 x 100000; one block per (n, d, h) row 65 and 87,
// and 4530 and 1440 (the chip idle but for eight blocks); so 58 and 82, 19 and
// 27.
// n / d = n m >> s for n < 2^31: 2^(s - 31) >= d, m = ceil(2^s / d)
struct Div {
  uint32_t m, s, d;
};
struct Item {
  int n, d, h, w, c;
};
// sizes of an output in items: 8-channel groups, W, H, D
struct Sizes32 {
  typedef uint32_t Index;
  Div c, w, h, d;
};
struct Sizes64 {
  typedef uint64_t Index;
  uint64_t c, w, h, d;
};
__device__ __forceinline__ uint32_t div_rem(uint32_t n, Div v, int &rem) {
  uint32_t const q = (uint32_t)(((uint64_t)n * v.m) >> v.s);
  rem = (int)(n - q * v.d);
  return q;
}
__device__ __forceinline__ uint64_t div_rem(uint64_t n, uint64_t v, int &rem) {
  rem = (int)(n % v);
  return n / v;
}
template <typename S>
__device__ __forceinline__ Item item_at(typename S::Index i, S const &z) {
  Item r;
  i = div_rem(i, z.c, r.c);
  r.c *= 8;
  i = div_rem(i, z.w, r.w);
  i = div_rem(i, z.h, r.h);
  r.n = (int)div_rem(i, z.d, r.d);
  return r;
}
#define ITEMS(idx, S, total)                                                        \
  for (typename S::Index idx = (typename S::Index)blockIdx.x * UT + threadIdx.x; idx < total; \
       idx += (typename S::Index)gridDim.x * UT)

// 2x2x2 max pool: y[n][d][h][w][c] over x[n][2d..][2h..][2w..][c]; arg holds
// the winning offset (first maximum in (a, b, e) order). D, H, W: of y
template <typename S>
__global__ __launch_bounds__(UT) void k_maxpool(uint16_t const *__restrict__ x,
                                                uint16_t *__restrict__ y,
                                                uint8_t *__restrict__ arg, int D, int H, int W,
                                                int C, S z, typename S::Index total) {
  ITEMS(idx, S, total) {
    Item const r = item_at(idx, z);
    float best[8];
    int barg[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      best[k] = -INFINITY;
      barg[k] = 0;
    }
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      int const a = o >> 2, b = (o >> 1) & 1, e = o & 1;
      int64_t const row = ((int64_t)r.n * 2 * D + 2 * r.d + a) * 2 * H + 2 * r.h + b;
      u16x8 const v = ld8(x + (row * 2 * W + 2 * r.w + e) * C + r.c);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float const f = bf2f(v[k]);
        if (f > best[k]) {
          best[k] = f;
          barg[k] = o;
        }
      }
    }
    u16x8 out;
    u8x8 ar;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      out[k] = f2bf(best[k]);
      ar[k] = (uint8_t)barg[k];
    }
    st8(y + (int64_t)idx * 8, out);
    *(u8x8 *)(arg + (int64_t)idx * 8) = ar;
  }
}

// gradient of the pooling, D, H, W: of dx. add (or NULL): a second gradient of
// the pooled tensor's input, its channels [c0, c0 + C) of Ca, added in fp32 and
// rounded once (as k_copy_channels mode 1 on the written dx)
template <typename S>
__global__ __launch_bounds__(UT) void k_maxpool_bwd(
    uint16_t const *__restrict__ dy, uint8_t const *__restrict__ arg, uint16_t *__restrict__ dx,
    int D, int H, int W, int C, uint16_t const *__restrict__ add, int Ca, int c0, S z,
    typename S::Index total) {
  ITEMS(idx, S, total) {
    Item const r = item_at(idx, z);
    int64_t const prow = ((int64_t)r.n * (D / 2) + r.d / 2) * (H / 2) + r.h / 2;
    int64_t const o = (prow * (W / 2) + r.w / 2) * C + r.c;
    int const mine = ((r.d & 1) << 2) | ((r.h & 1) << 1) | (r.w & 1);
    u16x8 const g = ld8(dy + o);
    u8x8 const a = *(u8x8 const *)(arg + o);
    u16x8 out;
#pragma unroll
    for (int k = 0; k < 8; ++k) out[k] = a[k] == mine ? g[k] : (uint16_t)0;
    if (add != nullptr) {
      int64_t const v = (((int64_t)r.n * D + r.d) * H + r.h) * W + r.w;
      u16x8 const s = ld8(add + v * Ca + c0 + r.c);
#pragma unroll
      for (int k = 0; k < 8; ++k) out[k] = f2bf(bf2f(s[k]) + bf2f(out[k]));
    }
    st8(dx + (int64_t)idx * 8, out);
  }
}

// y = [upsample(xu), xs]: the nearest x2 upsampling of xu (CU channels) and xs
// (CS channels) side by side, whole voxels of y [n][D][H][W][CU + CS] at a time
template <typename S>
__global__ __launch_bounds__(UT) void k_concat_up(uint16_t const *__restrict__ xu,
                                                  uint16_t const *__restrict__ xs,
                                                  uint16_t *__restrict__ y, int D, int H, int W,
                                                  int CU, int CS, S z, typename S::Index total) {
  ITEMS(idx, S, total) {
    Item const r = item_at(idx, z);
    int64_t const urow = ((int64_t)r.n * (D / 2) + r.d / 2) * (H / 2) + r.h / 2;
    int64_t const v = (((int64_t)r.n * D + r.d) * H + r.h) * W + r.w;
    uint16_t const *const q = r.c < CU ? xu + (urow * (W / 2) + r.w / 2) * CU + r.c
                                       : xs + v * CS + (r.c - CU);
    st8(y + (int64_t)idx * 8, ld8(q));
  }
}

// nearest x2 upsampling of x [n][D][H][W][C] into the channels [c0, c0 + C)
// of y [n][2D][2H][2W][Cy]
__global__ void k_upsample(uint16_t const *__restrict__ x, uint16_t *__restrict__ y, int N,
                           int D, int H, int W, int C, int Cy, int c0) {
  int const C8 = C / 8;
  int64_t const total = (int64_t)N * 8 * D * H * W * C8;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int const c = (int)(idx % C8) * 8;
    int64_t r = idx / C8;
    int const w = (int)(r % (2 * W));
    r /= 2 * W;
    int const h = (int)(r % (2 * H));
    r /= 2 * H;
    int const d = (int)(r % (2 * D));
    int const n = (int)(r / (2 * D));
    st8(y + ((((int64_t)n * 2 * D + d) * 2 * H + h) * 2 * W + w) * Cy + c0 + c,
        ld8(x + ((((int64_t)n * D + d / 2) * H + h / 2) * W + w / 2) * C + c));
  }
}

// gradient of the upsampling: dx[v][c] = sum of the 8 children's
// dy[..][c0 + c], in a fixed order; accumulated in fp32. D, H, W: of dx
template <typename S>
__global__ __launch_bounds__(UT) void k_upsample_bwd(uint16_t const *__restrict__ dy,
                                                     uint16_t *__restrict__ dx, int D, int H,
                                                     int W, int Cy, int c0, S z,
                                                     typename S::Index total) {
  ITEMS(idx, S, total) {
    Item const r = item_at(idx, z);
    float s[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) s[k] = 0.f;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      int const a = o >> 2, b = (o >> 1) & 1, e = o & 1;
      int64_t const row = ((int64_t)r.n * 2 * D + 2 * r.d + a) * 2 * H + 2 * r.h + b;
      u16x8 const g = ld8(dy + (row * 2 * W + 2 * r.w + e) * Cy + c0 + r.c);
#pragma unroll
      for (int k = 0; k < 8; ++k) s[k] += bf2f(g[k]);
    }
    u16x8 out;
#pragma unroll
    for (int k = 0; k < 8; ++k) out[k] = f2bf(s[k]);
    st8(dx + (int64_t)idx * 8, out);
  }
}

// channel slice copy: y[v][cy0 + c] = x[v][cx0 + c], c < C, v < nvox
// (mode 1: added to y, fp32 sum rounded once; mode 2: zero where
// gate[v][cy0 + c] <= 0)
__global__ void k_copy_channels(uint16_t const *__restrict__ x, uint16_t *__restrict__ y,
                                int64_t nvox, int Cx, int cx0, int Cy, int cy0, int C,
                                int mode, uint16_t const *__restrict__ gate) {
  int const C8 = C / 8;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < nvox * C8;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int64_t const v = idx / C8;
    int const c = (int)(idx - v * C8) * 8;
    u16x8 val = ld8(x + v * Cx + cx0 + c);
    if (mode == 1) {
      u16x8 const o = ld8(y + v * Cy + cy0 + c);
#pragma unroll
      for (int k = 0; k < 8; ++k) val[k] = f2bf(bf2f(val[k]) + bf2f(o[k]));
    } else if (mode == 2) {
      u16x8 const g = ld8(gate + v * Cy + cy0 + c);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (!(bf2f(g[k]) > 0.f)) val[k] = 0;
    }
    st8(y + v * Cy + cy0 + c, val);
  }
}

// fp32 field -> channel 0 of a bf16 tensor with C channels (others zero);
// one thread per voxel
__global__ void k_pack_input(float const *__restrict__ src, uint16_t *__restrict__ x,
                             int64_t nvox, int C, float scale) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nvox;
       v += (int64_t)gridDim.x * blockDim.x) {
    u16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    u16x8 first = z;
    first[0] = f2bf(src[v] * scale);
    st8(x + v * C, first);
    for (int c = 8; c < C; c += 8) st8(x + v * C + c, z);
  }
}

// channel 0 of a bf16 tensor -> fp32 field times scale (plus base if given)
__global__ void k_unpack_output(uint16_t const *__restrict__ y, float *__restrict__ dst,
                                float const *__restrict__ base, int64_t nvox, int C,
                                float scale) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nvox;
       v += (int64_t)gridDim.x * blockDim.x) {
    float const o = bf2f(y[v * C]) * scale;
    dst[v] = base ? base[v] + o : o;
  }
}

// L2 loss on channel 0: partial sums of (y - t)^2 per block, and
// dy = 2 (y - t) / nvox on channel 0 (zero elsewhere)
__global__ __launch_bounds__(UT) void k_l2_loss(uint16_t const *__restrict__ y,
                                               float const *__restrict__ t,
                                               uint16_t *__restrict__ dy,
                                               float *__restrict__ part, int64_t nvox, int C,
                                               float tscale) {
  __shared__ float red[UT];
  int64_t const v = (int64_t)blockIdx.x * UT + threadIdx.x;
  float e2 = 0.f;
  if (v < nvox) {
    float const e = bf2f(y[v * C]) - t[v] * tscale;
    e2 = e * e;
    uint16_t const g = f2bf(2.f * e / (float)nvox);
    if (C % 8 == 0) {
      u16x8 o = {g, 0, 0, 0, 0, 0, 0, 0};
      for (int c = 0; c < C; c += 8) {
        *(u16x8u *)(dy + v * C + c) = o;  // any bf16 pointer, as below
        o[0] = 0;
      }
    } else {
      dy[v * C] = g;
      for (int c = 1; c < C; ++c) dy[v * C + c] = 0;
    }
  }
  red[threadIdx.x] = e2;
  __syncthreads();
  for (int s = UT / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam on fp32 masters; writes the bf16 working copy (wb may be NULL)
__global__ void k_adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                       float const *__restrict__ g, uint16_t *__restrict__ wb, int len,
                       float lr, float b1, float b2, float eps, float c1, float c2) {
  int const i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= len) return;
  float const gi = g[i];
  float const mi = b1 * m[i] + (1.f - b1) * gi;
  float const vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float const wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

__global__ void k_to_bf16(float const *__restrict__ a, uint16_t *__restrict__ b, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = f2bf(a[i]);
}

__global__ void k_from_bf16(uint16_t const *__restrict__ b, float *__restrict__ a, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a[i] = bf2f(b[i]);
}

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
#define CONV_CASES(X) \
  X(16, 16) X(16, 32) X(32, 32) X(32, 64) X(64, 64) X(96, 32) X(48, 16) X(32, 16) \
  X(64, 32) X(32, 96) X(16, 48) X(64, 96) X(16, 64)

static inline int64_t blocks_for(int64_t n, int t) { return (n + t - 1) / t; }
// grid of the grid-stride elementwise kernels
static inline int64_t blocks_capped(int64_t n, int t) {
  int64_t const b = blocks_for(n, t);
  return b < (1 << 20) ? b : (1 << 20);
}

static Div div_by(uint32_t d) {
  Div v = {0, 31, d};
  while (((uint64_t)1 << (v.s - 31)) < d) ++v.s;
  v.m = (uint32_t)((((uint64_t)1 << v.s) + d - 1) / d);
  return v;
}

// a kernel of one thread per item of an [N][D][H][W][8 C8] output; small: its
// instance for fewer than 2^31 items, large: for any number
template <typename K, typename L, typename... A>
static int item_launch(char const *name, K small, L large, int N, int D, int H, int W, int C8,
                       void *stream, A... args) {
  int64_t const total = (int64_t)N * D * H * W * C8;
  dim3 const grid((unsigned)blocks_capped(total, UT));
  if (total <= 0) return 0;
  if (total < 0x7fffffff)
    return ulaunch(name, small, grid, dim3(UT), stream, args...,
                   Sizes32{div_by((uint32_t)C8), div_by((uint32_t)W), div_by((uint32_t)H),
                           div_by((uint32_t)D)},
                   (uint32_t)total);
  return ulaunch(name, large, grid, dim3(UT), stream, args...,
                 Sizes64{(uint64_t)C8, (uint64_t)W, (uint64_t)H, (uint64_t)D}, (uint64_t)total);
}

extern "C" {

// The kernels index within one d plane in 32-bit unsigned arithmetic (voxel
// index h * W + w in int, then times the channel count in uint32), so a
// plane's elements H * W * channels must stay below 2^32.
static int conv_shape_ok(int N, int D, int H, int W, int CI, int CO) {
  if (N < 1 || D < 1 || H < 1 || W < 1 || H > 65535 || (int64_t)N * D > 65535 ||
      (int64_t)H * W * (CI > CO ? CI : CO) >= ((int64_t)1 << 32)) {
    fprintf(stderr, "ERROR: convolution shape %d x %d x %d x %d unsupported\n", N, D, H, W);
    return 0;
  }
  return 1;
}

#define CONV_LAUNCH(a, b, u, p)                                                             \
  {                                                                                        \
    int const db = ConvDepth<b, u, p>::DB;                                                 \
    dim3 const grid((unsigned)((W + CT_W - 1) / CT_W), (unsigned)((H + CT_H - 1) / CT_H),  \
                    (unsigned)(N * ((D + db - 1) / db)));                                  \
    return ulaunch("conv3", k_conv3<a, b, u, p>, grid, dim3(UT), stream,                   \
                   (uint16_t const *)x, (uint16_t const *)xu, (uint16_t const *)wt,         \
                   (uint16_t const *)wcu, bias, (uint16_t const *)gate, (uint16_t *)y,       \
                   (uint16_t *)pool, D, H, W, mode);                                        \
  }

#define CONVS_DB 16
static int conv3s_launch(void const *x, void const *wt, float const *bias, void *y, void *pool,
                         int N, int D, int H, int W, int mode, void *stream) {
  dim3 const grid((unsigned)((W + CT_W - 1) / CT_W), (unsigned)((H + CT_H - 1) / CT_H),
                  (unsigned)(N * ((D + CONVS_DB - 1) / CONVS_DB)));
  if (mode & 8)
    return ulaunch("conv3s", k_conv3s<CONVS_DB, true>, grid, dim3(UT), stream,
                   (uint16_t const *)x, (uint16_t const *)wt, bias, (uint16_t *)y,
                   (uint16_t *)pool, D, H, W, mode);
  return ulaunch("conv3s", k_conv3s<CONVS_DB, false>, grid, dim3(UT), stream,
                 (uint16_t const *)x, (uint16_t const *)wt, bias, (uint16_t *)y,
                 (uint16_t *)pool, D, H, W, mode);
}

int agdu_conv3(void const *x, void const *wt, float const *bias, void const *gate, void *y,
               int N, int D, int H, int W, int CI, int CO, int mode, void *stream) {
  void const *const xu = NULL;
  void const *const wcu = NULL;
  void *const pool = NULL;
  mode &= 7;
  if (!conv_shape_ok(N, D, H, W, CI, CO)) return 1;
  // 16 -> 16 without the gradient's gate: the streaming form
  if (CI == 16 && CO == 16 && !(mode & 4))
    return conv3s_launch(x, wt, bias, y, NULL, N, D, H, W, mode, stream);
#define CC(a, b) \
  if (CI == a && CO == b) CONV_LAUNCH(a, b, 0, false)
  CONV_CASES(CC)
#undef CC
  fprintf(stderr, "ERROR: no convolution kernel for %d -> %d channels\n", CI, CO);
  return 1;
}

#define CAT_CASES(X) X(32, 16, 16) X(64, 32, 32)

/* agdu_conv3 that also writes the 2x2x2 max pooling of its output (the
   values agdu_maxpool gives, without the arg), for the layers whose blocks
   hold whole plane pairs */
int agdu_conv3_pool(void const *x, void const *wt, float const *bias, void *y, void *pool,
                    int N, int D, int H, int W, int CI, int CO, int mode, void *stream) {
  void const *const xu = NULL;
  void const *const wcu = NULL;
  void const *const gate = NULL;
  if (!conv_shape_ok(N, D, H, W, CI, CO)) return 1;
  if ((D | H | W) & 1 || pool == NULL) {
    fprintf(stderr, "ERROR: pooling needs even sizes and an output, got %d x %d x %d\n", D, H,
            W);
    return 1;
  }
  mode = (mode & 3) | 8;
  if (CI == 16 && CO == 16) return conv3s_launch(x, wt, bias, y, pool, N, D, H, W, mode, stream);
#define CP(a, b) \
  if (CI == a && CO == b && ConvDepth<b, 0>::DB % 2 == 0) CONV_LAUNCH(a, b, 0, false)
  CONV_CASES(CP)
#undef CP
  fprintf(stderr, "ERROR: no pooling convolution kernel for %d -> %d channels\n", CI, CO);
  return 1;
}

int agdu_conv3_cat(void const *xu, void const *x, void const *wt, float const *bias,
                   void const *gate, void *y, int N, int D, int H, int W, int CU, int CS,
                   int CO, int mode, void *stream) {
  void const *const wcu = NULL;
  void *const pool = NULL;
  mode &= 7;
  if (!conv_shape_ok(N, D, H, W, CU + CS, CO)) return 1;
  if ((D | H | W) & 1) {
    fprintf(stderr, "ERROR: upsampled concatenation needs even sizes, got %d x %d x %d\n", D,
            H, W);
    return 1;
  }
#define CT(u, c, o) \
  if (CU == u && CS == c && CO == o) CONV_LAUNCH(u + c, o, u, false)
  CAT_CASES(CT)
#undef CT
  fprintf(stderr, "ERROR: no concatenating convolution for %d + %d -> %d channels\n", CU, CS,
          CO);
  return 1;
}

int agdu_up_weights(void const *wt, void *wcu, int CI, int CO, int CU, void *stream) {
  if (CU < 16 || CU % 16 || CU >= CI || CO < 16 || CO % 16) {
    fprintf(stderr, "ERROR: combined taps for %d of %d -> %d channels unsupported\n", CU, CI,
            CO);
    return 1;
  }
  int64_t const n = (int64_t)48 * CO * CU;
  return ulaunch("up_weights", k_up_weights, dim3((unsigned)blocks_capped(n, UT)), dim3(UT),
                 stream, (uint16_t const *)wt, (uint16_t *)wcu, CI, CO, CU);
}

int agdu_conv3_up(void const *xu, void const *x, void const *wt, void const *wcu,
                  float const *bias, void const *gate, void *y, int N, int D, int H, int W,
                  int CU, int CS, int CO, int mode, void *stream) {
  if (!conv_shape_ok(N, D, H, W, CU + CS, CO)) return 1;
  if ((D | H | W) & 1) {
    fprintf(stderr, "ERROR: upsampled concatenation needs even sizes, got %d x %d x %d\n", D,
            H, W);
    return 1;
  }
  if (wcu == NULL) {
    fprintf(stderr, "ERROR: combined taps missing\n");
    return 1;
  }
  void *const pool = NULL;
  mode &= 7;
#define CT(u, c, o) \
  if (CU == u && CS == c && CO == o) CONV_LAUNCH(u + c, o, u, true)
  CAT_CASES(CT)
#undef CT
  fprintf(stderr, "ERROR: no concatenating convolution for %d + %d -> %d channels\n", CU, CS,
          CO);
  return 1;
}

int agdu_conv_in(float const *src, void const *wt, int wci, float const *bias, void *y, int N,
                 int D, int H, int W, float scale, void *stream) {
  if (!conv_shape_ok(N, D, H, W, 16, 16)) return 1;
  if (wci < 1) {
    fprintf(stderr, "ERROR: first-layer weights must have input channels, got %d\n", wci);
    return 1;
  }
  dim3 const grid((unsigned)((W + CT_W - 1) / CT_W), (unsigned)((H + CT_H - 1) / CT_H),
                  (unsigned)(N * ((D + FDB - 1) / FDB)));
  return ulaunch("conv_first", k_conv_first, grid, dim3(UT), stream, src,
                 (uint16_t const *)wt, wci, bias, (uint16_t *)y, D, H, W, scale);
}

int agdu_conv_out(void const *x, void const *wt, int wco, float const *bias, float const *base,
                  float *dst, int N, int D, int H, int W, float unscale, void *stream) {
  if (!conv_shape_ok(N, D, H, W, 16, 16)) return 1;
  if (wco < 1) {
    fprintf(stderr, "ERROR: head with %d output channels unsupported\n", wco);
    return 1;
  }
  dim3 const grid((unsigned)((W + CT_W - 1) / CT_W), (unsigned)((H + CT_H - 1) / CT_H),
                  (unsigned)(N * ((D + HDB - 1) / HDB)));
  return ulaunch("conv_head", k_conv_head, grid, dim3(UT), stream, (uint16_t const *)x,
                 (uint16_t const *)wt, wco, bias, base, dst, D, H, W, unscale);
}

int agdu_flip_weights(void const *wt, void *wtt, int CI, int CO, void *stream) {
  int const total = 27 * CI * CO;
  return ulaunch("flip_weights", k_flip_weights, dim3((unsigned)blocks_for(total, UT)),
                 dim3(UT), stream, (uint16_t const *)wt, (uint16_t *)wtt, CI, CO);
}

// the channel pairs of the network's layers (and their input gradients), and
// the share of 2048 blocks that cuts a pair's rows into blocks
#define WGRAD_CASES(X) \
  X(16, 16, 3) X(16, 32, 3) X(32, 32, 3) X(48, 16, 3) X(32, 16, 3) X(32, 64, 9) X(64, 64, 9) \
  X(96, 32, 9) X(64, 32, 9) X(16, 64, 3)

// launch shape of the weight gradient: tile pairs, rows per row chunk and row
// chunks (each of 3 pairs blocks); 0 when the channel pair has no kernel
static int wgrad_plan(int N, int D, int H, int W, int CI, int CO, int *pairs, int *rb,
                      int64_t *nblk) {
  int share = 0;
#define WC(a, b, k) \
  if (CI == a && CO == b) share = k;
  WGRAD_CASES(WC)
#undef WC
  if (share == 0) return 0;
  *pairs = (CI / 16) * (CO / 16);
  int64_t const rows = (int64_t)N * D * H;
  int64_t const nwc = (W + 63) / 64;
  int64_t const target = 2048 / share;
  int64_t r = (rows * nwc + target - 1) / target;
  if (r < 1) r = 1;
  *rb = (int)r;
  *nblk = nwc * ((rows + r - 1) / r);
  return 1;
}

int64_t agdu_wgrad_part_len(int N, int D, int H, int W, int CI, int CO) {
  int pairs, rb;
  int64_t nblk;
  if (!wgrad_plan(N, D, H, W, CI, CO, &pairs, &rb, &nblk)) return -1;
  return nblk * (27 * CI * CO + CO);
}

int agdu_conv3_wgrad(void const *x, void const *dy, float *part, float *dw, float *db, int N,
                     int D, int H, int W, int CI, int CO, void *stream) {
  int pairs, rb;
  int64_t nblk;
  if (N < 1 || D < 1 || H < 1 || W < 1 ||
      !wgrad_plan(N, D, H, W, CI, CO, &pairs, &rb, &nblk) ||
      3 * pairs * nblk > 0x7fffffff) {
    fprintf(stderr, "ERROR: weight gradient for %d -> %d channels, %d x %d x %d x %d "
                    "unsupported\n", CI, CO, N, D, H, W);
    return 1;
  }
  int const len = 27 * CI * CO;
  float *const bpart = part + nblk * len;
  if (ulaunch("conv3_wgrad", k_conv3_wgrad, dim3((unsigned)(3 * pairs * nblk)), dim3(WG_T),
              stream, (uint16_t const *)x, (uint16_t const *)dy, part, db ? bpart : (float *)0, D,
              H, W, CI, CO, (int64_t)N * D * H, rb))
    return 1;
  return ulaunch("reduce_parts", k_reduce_parts,
                 dim3((unsigned)((len + 15) / 16 + (db ? CO / 16 : 0))), dim3(UT), stream,
                 (float const *)part, dw, (int)nblk, len, (float const *)bpart, db, CO);
}

int agdu_maxpool(void const *x, void *y, void *arg, int N, int D, int H, int W, int C,
                 void *stream) {
  if ((D | H | W) & 1) {
    fprintf(stderr, "ERROR: max pooling needs even sizes, got %d x %d x %d\n", D, H, W);
    return 1;
  }
  if (C % 8) {
    fprintf(stderr, "ERROR: channel count %d is not a multiple of 8\n", C);
    return 1;
  }
  return item_launch("maxpool", k_maxpool<Sizes32>, k_maxpool<Sizes64>, N, D / 2, H / 2, W / 2,
                     C / 8, stream, (uint16_t const *)x, (uint16_t *)y, (uint8_t *)arg, D / 2,
                     H / 2, W / 2, C);
}

int agdu_maxpool_bwd_add(void const *dy, void const *arg, void const *add, int Ca, int c0,
                         void *dx, int N, int D, int H, int W, int C, void *stream) {
  if ((D | H | W) & 1) {
    fprintf(stderr, "ERROR: max pooling needs even sizes, got %d x %d x %d\n", D, H, W);
    return 1;
  }
  if (C % 8) {
    fprintf(stderr, "ERROR: channel count %d is not a multiple of 8\n", C);
    return 1;
  }
  if (add != NULL && ((Ca | c0) % 8 || c0 < 0 || c0 + C > Ca)) {
    fprintf(stderr, "ERROR: added channels %d at %d of %d unsupported\n", C, c0, Ca);
    return 1;
  }
  return item_launch("maxpool_bwd", k_maxpool_bwd<Sizes32>, k_maxpool_bwd<Sizes64>, N, D, H, W,
                     C / 8, stream, (uint16_t const *)dy, (uint8_t const *)arg, (uint16_t *)dx, D,
                     H, W, C, (uint16_t const *)add, Ca, c0);
}

int agdu_maxpool_bwd(void const *dy, void const *arg, void *dx, int N, int D, int H, int W,
                     int C, void *stream) {
  return agdu_maxpool_bwd_add(dy, arg, NULL, 0, 0, dx, N, D, H, W, C, stream);
}

int agdu_concat_up(void const *xu, void const *xs, void *y, int N, int D, int H, int W, int CU,
                   int CS, void *stream) {
  if ((D | H | W) & 1) {
    fprintf(stderr, "ERROR: upsampling needs even sizes, got %d x %d x %d\n", D, H, W);
    return 1;
  }
  if ((CU | CS) % 8) {
    fprintf(stderr, "ERROR: concatenating %d and %d channels unsupported\n", CU, CS);
    return 1;
  }
  return item_launch("concat_up", k_concat_up<Sizes32>, k_concat_up<Sizes64>, N, D, H, W,
                     (CU + CS) / 8, stream, (uint16_t const *)xu, (uint16_t const *)xs,
                     (uint16_t *)y, D, H, W, CU, CS);
}

int agdu_upsample(void const *x, void *y, int N, int D, int H, int W, int C, int Cy, int c0,
                  void *stream) {
  if ((C | Cy | c0) % 8 || c0 + C > Cy) {
    fprintf(stderr, "ERROR: upsampling channels %d at %d of %d unsupported\n", C, c0, Cy);
    return 1;
  }
  int64_t const total = (int64_t)N * 8 * D * H * W * (C / 8);
  return ulaunch("upsample", k_upsample, dim3((unsigned)blocks_capped(total, UT)), dim3(UT),
                 stream, (uint16_t const *)x, (uint16_t *)y, N, D, H, W, C, Cy, c0);
}

int agdu_upsample_bwd(void const *dy, void *dx, int N, int D, int H, int W, int C, int Cy,
                      int c0, void *stream) {
  if ((C | Cy | c0) % 8 || c0 + C > Cy) {
    fprintf(stderr, "ERROR: upsampling channels %d at %d of %d unsupported\n", C, c0, Cy);
    return 1;
  }
  return item_launch("upsample_bwd", k_upsample_bwd<Sizes32>, k_upsample_bwd<Sizes64>, N, D, H,
                     W, C / 8, stream, (uint16_t const *)dy, (uint16_t *)dx, D, H, W, Cy, c0);
}

int agdu_copy_channels(void const *x, void *y, int64_t nvox, int Cx, int cx0, int Cy,
                       int cy0, int C, int mode, void const *gate, void *stream) {
  if ((Cx | cx0 | Cy | cy0 | C) % 8 || cx0 + C > Cx || cy0 + C > Cy) {
    fprintf(stderr, "ERROR: channel copy %d at %d of %d -> %d of %d unsupported\n", C, cx0, Cx,
            cy0, Cy);
    return 1;
  }
  return ulaunch("copy_channels", k_copy_channels,
                 dim3((unsigned)blocks_capped(nvox * (C / 8), UT)), dim3(UT), stream,
                 (uint16_t const *)x, (uint16_t *)y, nvox, Cx, cx0, Cy, cy0, C, mode,
                 (uint16_t const *)gate);
}

int agdu_pack_input(float const *src, void *x, int64_t nvox, int C, float scale,
                    void *stream) {
  if (C % 8) {
    fprintf(stderr, "ERROR: channel count %d is not a multiple of 8\n", C);
    return 1;
  }
  return ulaunch("pack_input", k_pack_input, dim3((unsigned)blocks_capped(nvox, UT)),
                 dim3(UT), stream, src, (uint16_t *)x, nvox, C, scale);
}

int agdu_unpack_output(void const *y, float *dst, float const *base, int64_t nvox, int C,
                       float scale, void *stream) {
  return ulaunch("unpack_output", k_unpack_output, dim3((unsigned)blocks_capped(nvox, UT)),
                 dim3(UT), stream, (uint16_t const *)y, dst, base, nvox, C, scale);
}

int agdu_l2_loss(void const *y, float const *t, void *dy, float *part, int64_t nvox, int C,
                 float tscale, void *stream) {
  return ulaunch("l2_loss", k_l2_loss, dim3((unsigned)blocks_for(nvox, UT)), dim3(UT),
                 stream, (uint16_t const *)y, t, (uint16_t *)dy, part, nvox, C, tscale);
}

int64_t agdu_loss_parts(int64_t nvox) { return blocks_for(nvox, UT); }

int agdu_adam(float *w, float *m, float *v, float const *g, void *wb, int len, float lr,
              float b1, float b2, float eps, int step, void *stream) {
  float const c1 = 1.f - powf(b1, (float)step);
  float const c2 = 1.f - powf(b2, (float)step);
  return ulaunch("adam", k_adam, dim3((unsigned)blocks_for(len, UT)), dim3(UT), stream, w, m,
                 v, g, (uint16_t *)wb, len, lr, b1, b2, eps, c1, c2);
}

int agdu_to_bf16(float const *a, void *b, int64_t n, void *stream) {
  return ulaunch("to_bf16", k_to_bf16, dim3((unsigned)blocks_capped(n, UT)), dim3(UT), stream,
                 a, (uint16_t *)b, n);
}

int agdu_from_bf16(void const *b, float *a, int64_t n, void *stream) {
  return ulaunch("from_bf16", k_from_bf16, dim3((unsigned)blocks_capped(n, UT)), dim3(UT),
                 stream, (uint16_t const *)b, a, n);
}

}  // extern "C"
