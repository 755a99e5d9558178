// Launches on the library stream, shared by the files that hold its kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "agd_gpu.h"

#define NTHR 256
#define TIME_SPLIT_BLOCKS 1536

// the library stream; *a: the start event when kernels are timed, else null
hipStream_t agd_launch_begin(hipEvent_t *a);
// checks the launch and, when timed, keeps the pair of events under name
int agd_launch_end(char const *name, hipEvent_t a);

template <typename K, typename... Args>
static int launch(char const *name, K kernel, dim3 grid, dim3 block, size_t lds,
                  Args... args) {
  hipEvent_t a;
  if (grid.x == 0 || grid.y == 0 || grid.z == 0) return 0;
  hipStream_t const s = agd_launch_begin(&a);
  hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
  return agd_launch_end(name, a);
}

// Blocks go to the eight XCDs in turn (block b runs on XCD b mod 8, each
// XCD with its own L2). This bijection of [0, n) gives XCD x a contiguous
// run of the n work items instead.
__device__ __forceinline__ int xcd_chunk(int b, int n) {
  int const q = n >> 3, r = n & 7, x = b & 7, i = b >> 3;
  return x * q + min(x, r) + i;
}

// the larger of two non-negative floats, or a NaN if there is one (their
// bits order that way)
__device__ __forceinline__ float max_bits(float a, float b) {
  return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
}

// soft threshold x (|x| - lamb) / |x| when |x| > lamb, else 0; one rounding
// order in every kernel that inlines it
__device__ __forceinline__ float2 soft(float2 v, float lamb) {
  float const a = fmaf(v.x, v.x, v.y * v.y);
  float const s = fmaxf(fmaf(-lamb, __builtin_amdgcn_rsqf(a), 1.f), 0.f);
  return make_float2(v.x * s, v.y * s);
}
// x - alpha g
__device__ __forceinline__ float2 step(float2 x, float alpha, float2 g) {
  return make_float2(fmaf(-alpha, g.x, x.x), fmaf(-alpha, g.y, x.y));
}

// units of class c within the launch's window range: [*first, *first + n)
static inline int class_range(AgdDev const *g, AgdClass const &c, int *first) {
  int const a = c.wpos[g->w0], b = c.wpos[g->w1];
  *first = c.begin + a;
  return b - a;
}

// the specialised kernels may use up to the CU's 160 KB of LDS: set once per
// kernel instance, on its first launch
static inline int allow_lds(void const *f) {
  (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  (void)hipGetLastError();
  return 1;
}

// the card's compute units, and the blocks of `threads` threads and lds bytes of
// dynamic LDS that it holds at once of a kernel (asked once per instance)
int agd_compute_units(void);
int agd_resident(void const *kernel, int threads, size_t lds);

// Most runs that a launch of n time blocks of class c splits each block's time
// windows into (grid y), at least `least` time windows to a run. A block's
// time windows are a serial chain, so below TIME_SPLIT_BLOCKS blocks (six
// per CU) the chip waits on it: 30 blocks of 9 time windows (256 x 1024
// line, windows 32 x 256) took 27 us forward and 34 adjoint as one run each
// and take 15 and 11 split, 236 blocks of 14 (1510 x 1251 line, windows 50 x
// 200) 143 and 169 and 36 and 33. Runs given by AGD_TIME_TW are left as they
// are.
static inline int time_split(AgdDev const *g, AgdClass const &c, int n, int least) {
  if (!g->split_time) return 1;
  int const want = (TIME_SPLIT_BLOCKS + n - 1) / n, most = c.ntw / least;
  int const r = want < most ? want : most;
  return r > 1 ? r : 1;
}

// The forward's runs, each of which repeats the time window before it for its
// carry: of the counts up to the most, the one whose rounds of resident blocks
// take the fewest time windows one after the other. By the count of blocks
// alone, 1280 runs of 2 of 4 time windows (40 x 96 x 384 in windows of 16 x 32 x
// 256, 768 blocks resident) took 29 us, the 640 blocks as one run each 25; the
// line of 1510 x 1251 43 us in runs of 2, 36 in runs of 3; 1800 x 2000 in windows
// of 18 x 500 197 and, as one run each, 148.
static inline int time_split_fwd(AgdDev const *g, AgdClass const &c, int n, int resident) {
  int const most = time_split(g, c, n, 2);
  int best = 1;
  int64_t best_cost = 0;
  for (int r = 1; r <= most; ++r) {
    int64_t const rounds = ((int64_t)n * r + resident - 1) / resident;
    int64_t const cost = rounds * ((c.ntw + r - 1) / r + (r > 1));
    if (r == 1 || cost < best_cost) {
      best = r;
      best_cost = cost;
    }
  }
  return best;
}
