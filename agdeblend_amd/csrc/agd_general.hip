// Transforms of any window size, up to four space dims (HIP kernels and their
// launchers, declared in agd_general.h).
//
// A patch whose size is not a multiple of its half windows gets windows one
// or a few samples longer than asked for, so padded lengths such as 23, 42
// or 43 are the usual case, not the exception. These kernels take the
// lengths at run time. Every 1-D transform is a line held by one thread in
// registers (Line): the DFT of P values on the pairs
//   a_k = x_k + x_{P-k},  b_k = x_k - x_{P-k},   0 < k < P / 2,
//   X_q, X_{P-q} = (x_0 + (-1)^q x_{P/2} + sum a_k cos(2 pi q k / P))
//                  +- i S sum b_k sin(2 pi q k / P),
// i.e. P^2 real multiply-adds for P complex outputs, half of the plain sum,
// with coefficients that are the same for every thread and come through
// the scalar cache as instruction operands. No roots, divisions or LDS
// traffic inside a line, and no dependence on how P factors. Lengths without
// a prime factor above 13 take a register FFT instead (codelets). Where that
// FFT's registers would leave few waves (above 33), P = A B folds into two
// short ones in place (FOLD).
//
// Measured (MI355X) on a 45 x 333 x 1500 volume in two patches, windows of
// 17-18 x 24-25 x 200 (P = 22, 23 x 30, 32, Pt = 250; model 1.15 GB), us per
// iteration: spatial transforms and update 15480 by the LDS-resident kernels
// (radix passes through LDS with table roots, forward and adjoint apart) ->
// 1640 lines as above -> 1620 with the codelets -> 990 with reciprocals for
// integer divisions (1000 with last tiles as wide as their traces); it moves
// 3.9 GB, 820 us at this card's copy rate. Time transforms 1460 and 1670 ->
// 480 and 500 -> 291 and 278. Prefetching the model's values ahead of the
// transforms changed nothing (the lines' registers are worth more as waves).
#include <hip/hip_runtime.h>

#include "agd_fft.h"
#include "agd_general.h"
#include "agd_launch.h"

namespace agdgen {

// coefficient tables are read through the scalar cache (constant address
// space, block-uniform addresses)
typedef float __attribute__((address_space(4))) cfloat;
__device__ __forceinline__ cfloat const *uniform(float const *p, int off) {
  return (cfloat const *)(uintptr_t)(p + __builtin_amdgcn_readfirstlane(off));
}

// rows of the coefficient table of length P: for q = 1 .. (P - 1) / 2 the
// pairs cos, sin(2 pi q k / P), k = 1 .., padded with zeros to whole groups
// of 4 pairs (built by the host, dft_get)
__device__ __forceinline__ int table_row(int P) { return 2 * (((P - 1) / 2 + 3) & ~3); }

// One line's inputs as the pairs a, b (and x_0, x_{P/2}).
template <int HB>
struct Line {
  float2 a[HB], b[HB], x0, xh;

  // the line ln[k st], k < P: the inputs k >= nin are zero. P - 1 <= 2 HB.
  // Everything but ln is uniform over the block.
  __device__ __forceinline__ void load(float2 const *ln, int st, int P, int nin) {
    int const h = (P - 1) >> 1;
    x0 = ln[0];
    xh = make_float2(0.f, 0.f);
    if (!(P & 1) && P / 2 < nin) xh = ln[(P / 2) * st];
#pragma unroll
    for (int c = 0; c < HB; c += 4) {
      if (c < h) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          int const k = c + u + 1;
          // clamped loads, values outside the line or its inputs unused
          float2 const p = ln[min(k, nin - 1) * st];
          float2 const m = ln[max(0, min(P - k, nin - 1)) * st];
          bool const hp = k <= h && k < nin, hm = k <= h && P - k < nin;
          float2 const x = make_float2(hp ? p.x : 0.f, hp ? p.y : 0.f);
          float2 const y = make_float2(hm ? m.x : 0.f, hm ? m.y : 0.f);
          a[c + u] = make_float2(x.x + y.x, x.y + y.y);
          b[c + u] = make_float2(x.x - y.x, x.y - y.y);
        }
      }
    }
  }

  // DFT of sign S: the outputs of part `part` of `parts` (uniform over the
  // wave) below nout to out(q, X_q)
  template <int S, class Out>
  __device__ __forceinline__ void dft(int P, int nout, cfloat const *tab, int part, int parts,
                                      Out const &out) const {
    int const h = (P - 1) >> 1;
    if (part == 0) {
      float2 sum = x0, alt = x0;
#pragma unroll
      for (int c = 0; c < HB; c += 4) {
        if (c < h) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            sum.x += a[c + u].x;
            sum.y += a[c + u].y;
            if (u & 1) {  // k = c + u + 1 is even
              alt.x += a[c + u].x;
              alt.y += a[c + u].y;
            } else {
              alt.x -= a[c + u].x;
              alt.y -= a[c + u].y;
            }
          }
        }
      }
      out(0, make_float2(sum.x + xh.x, sum.y + xh.y));
      if (!(P & 1) && P / 2 < nout) {
        float const s = (P / 2) & 1 ? -1.f : 1.f;
        out(P / 2, make_float2(alt.x + s * xh.x, alt.y + s * xh.y));
      }
    }
    int const row = table_row(P), q1 = 1 + h * (part + 1) / parts;
    int q = 1 + h * part / parts;
    for (tab += (q - 1) * row; q < q1; ++q, tab += row) {
      float const s = q & 1 ? -1.f : 1.f;
      float cr = x0.x + s * xh.x, ci = x0.y + s * xh.y, sr = 0.f, si = 0.f;
#pragma unroll
      for (int c = 0; c < HB; c += 4) {
        if (c < h) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            float const co = tab[2 * (c + u)], sn = tab[2 * (c + u) + 1];
            cr += co * a[c + u].x;
            ci += co * a[c + u].y;
            sr += sn * b[c + u].x;
            si += sn * b[c + u].y;
          }
        }
      }
      if (S < 0) {
        sr = -sr;
        si = -si;
      }
      // C +- i S (sr + i si)
      if (q < nout) out(q, make_float2(cr - si, ci + sr));
      if (P - q < nout) out(P - q, make_float2(cr + si, ci - sr));
    }
  }
};

// The DFTs of `total` lines in place, 64 to a wave: line l at at(l), output
// q of it through put(l, line, q, value). Up to 64 (128) lines are shared by
// four (two) waves, each computing a part of every line's outputs, so that
// short batches still use the whole block; a barrier then separates the
// waves' loads from the first output. Ends with a barrier.
template <int HB, int S, class At, class Put>
__device__ __forceinline__ void block_lines(int total, int st, int P, int nin, int nout,
                                            cfloat const *tab, At const &at, Put const &put) {
  int const lane = threadIdx.x & 63;
  int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Line<HB> ln;
  if (total <= 128) {
    int const parts = total <= 64 ? 4 : 2, part = total <= 64 ? wave : wave >> 1;
    int const l = total <= 64 ? lane : (wave & 1) * 64 + lane;
    auto const z = at(min(l, total - 1));
    ln.load(z.p, st, P, nin);
    __syncthreads();
    if (l < total)
      ln.template dft<S>(P, nout, tab, part, parts, [&](int q, float2 v) { put(z, q, v); });
  } else {
    for (int l = threadIdx.x; l < total; l += 256) {
      auto const z = at(l);
      ln.load(z.p, st, P, nin);
      ln.template dft<S>(P, nout, tab, 0, 1, [&](int q, float2 v) { put(z, q, v); });
    }
  }
  __syncthreads();
}

// a / d of small non-negative integers (a < 2^14 or so), inv = 1.f / d
__device__ __forceinline__ int quot(int a, float inv) {
  return (int)(((float)a + 0.5f) * inv);
}

// ---------------------------------------------------------------------------
// Spatial transforms: one block holds nk time-frequency planes of one (window,
// time window) in LDS, each a padded [P_0]..[P_{n-1}] array with rows of
// (P_{n-1} | 1) values (an odd pitch: the lanes of a row transform read
// distinct banks). Lines along a dim are transformed in place, one thread per
// line; the model is read and written once, coalesced, between the adjoint's
// dims (last to first) and the next forward's (first to last).
// ---------------------------------------------------------------------------
typedef int i4 __attribute__((ext_vector_type(AGD_MAXSP)));
struct Planes {
  int nsp, rows, pitch, rp;  // rows of a plane, row pitch, values of a plane
  i4 ext, str, P, W, A;      // per space dim (A: lines' first factor)
};

// a[i], uniform, without indexed registers
__device__ __forceinline__ int pick(i4 a, int i) {
  static_assert(AGD_MAXSP == 4, "four space dims");
  return i == 0 ? a.x : i == 1 ? a.y : i == 2 ? a.z : a.w;
}

// Padded lengths with a register codelet: no prime factor above 13, where the
// factored transform takes a third to a fifth of P^2 multiply-adds. The
// codelet knows the window length (W = 4 P / 5, rounded down: P = ceil(5 W /
// 4)): S < 0 reads W values and writes P, S > 0 the other way.
template <int P, int S>
__device__ __forceinline__ void codelet(float2 *ln, int st) {
  constexpr int W = P * 4 / 5, NIN = S < 0 ? W : P, NOUT = S < 0 ? P : W;
  float2 v[P];
#pragma unroll
  for (int k = 0; k < P; ++k) v[k] = k < NIN ? ln[k * st] : make_float2(0.f, 0.f);
  agdfft::fft<P, S>(v);
#pragma unroll
  for (int k = 0; k < NOUT; ++k) ln[k * st] = v[k];
}
// codelet P of the list Ps run on every line, or false
template <int S, class At>
__device__ __forceinline__ bool codelets(int, int, int, At const &) {
  return false;
}
template <int S, int N, int... Ps, class At>
__device__ __forceinline__ bool codelets(int P, int total, int st, At const &at) {
  if (P == N) {
    for (int l = threadIdx.x; l < total; l += 256) codelet<N, S>(at(l).p, st);
    __syncthreads();
    return true;
  }
  return codelets<S, Ps...>(P, total, st, at);
}

// The two phases of a folded line (lines): `total` lines at(i), each
// B (A) short lines, threads over (short line, line). rt[m] = exp(-2 pi i m /
// P).
template <int S, class At>
__device__ __forceinline__ void fold_a(int, int, int, float, int, int, At const &, float2 const *) {}
template <int S, int N, int... Ns, class At>
__device__ __forceinline__ void fold_a(int A, int B, int total, float it, int st, int nin,
                                       At const &at, float2 const *rt) {
  if (A != N) {
    fold_a<S, Ns...>(A, B, total, it, st, nin, at, rt);
    return;
  }
  int l = threadIdx.x, sb = B * st;
  asm volatile("" : "+v"(l), "+s"(sb));
  for (; l < total * B; l += 256) {
    int const r = quot(l, it);
    float2 *const z = at(l - r * total).p + r * st;
    float2 v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = r + k * B < nin ? z[k * sb] : make_float2(0.f, 0.f);
    agdfft::fft<N, S>(v);
    asm volatile("" : "+s"(sb) : : "memory");
#pragma unroll
    for (int q = 0; q < N; ++q) {
      float2 w = rt[q * r];
      if (S > 0) w.y = -w.y;
      z[q * sb] = q == 0 ? v[q] : agdfft::c_mul(v[q], w);
    }
  }
}
template <int S, class At>
__device__ __forceinline__ void fold_b(int, int, int, float, int, int, At const &) {}
template <int S, int N, int... Ns, class At>
__device__ __forceinline__ void fold_b(int A, int B, int total, float it, int st, int nout,
                                       At const &at) {
  if (B != N) {
    fold_b<S, Ns...>(A, B, total, it, st, nout, at);
    return;
  }
  // at most AGD_LINES_VALUES / N short lines
  constexpr int R = (AGD_LINES_VALUES / N + 255) / 256;
  int l0 = threadIdx.x, sa = A * st;
  asm volatile("" : "+v"(l0), "+s"(st));
  float2 v[R][N];
#pragma unroll
  for (int c = 0; c < R; ++c) {
    int const l = l0 + 256 * c;
    if (l < total * A) {
      int const n1 = quot(l, it);
      float2 const *const z = at(l - n1 * total).p + n1 * N * st;
#pragma unroll
      for (int k = 0; k < N; ++k) v[c][k] = z[k * st];
      agdfft::fft<N, S>(v[c]);
    }
  }
  __syncthreads();
  asm volatile("" : "+v"(l0), "+s"(sa));
#pragma unroll
  for (int c = 0; c < R; ++c) {
    int const l = l0 + 256 * c;
    if (l < total * A) {
      int const n1 = quot(l, it);
      float2 *const z = at(l - n1 * total).p + n1 * st;
#pragma unroll
      for (int k = 0; k < N; ++k)
        if (n1 + k * A < nout) z[k * sa] = v[c][k];
    }
  }
}

// transforms every line along dim d of the nk planes in place; the other
// dims run over their current extents g.ext
template <int HB, bool FOLD, int S>
__device__ __forceinline__ void lines(float2 *sm, Planes &g, int nk, int d, int nin, int nout,
                                      cfloat const *tab, float2 const *rt) {
  int cnt = 1;
#pragma unroll
  for (int e = 0; e < AGD_MAXSP; ++e)
    if (e < g.nsp && e != d) cnt *= g.ext[e];
  int const total = nk * cnt, st = pick(g.str, d), P = pick(g.P, d);
  float const inv = 1.f / (float)cnt;
  struct At {
    float2 *p;
  };
  auto const at = [&](int l) {
    int const k = quot(l, inv);
    int r = l - k * cnt, off = k * g.rp;
#pragma unroll
    for (int e = AGD_MAXSP - 1; e >= 0; --e) {
      if (e < g.nsp && e != d) {
        int const q = quot(r, 1.f / (float)g.ext[e]);
        off += (r - q * g.ext[e]) * g.str[e];
        r = q;
      }
    }
    return At{sm + off};
  };
  // P = A B in place: A-point lines over k1 (k = k1 B + k2), twiddle,
  // then B-point lines over k2, whose outputs n = n1 + A n2 go to their
  // natural places once every thread has read its inputs
  // (1-D lines of 64 on 59 windows of 51 x 126: one FFT in 228 registers
  // left 8 waves to a CU, three of four idle, 88 us; now 58, for 27 at
  // the cached copy rate; the block's four barriers bound it)
  int const A = pick(g.A, d), B = quot(P, 1.f / (float)A);
  auto const fold = [&] {
    float const it = 1.f / (float)total;
    fold_a<S, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>(A, B, total, it, st, nin, at, rt);
    __syncthreads();
    fold_b<S, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>(A, B, total, it, st, nout, at);
    if constexpr (HB > 0) fold_b<S, 25>(A, B, total, it, st, nout, at);
    __syncthreads();
  };
  if constexpr (HB == 0) {
    if (!codelets<S, 2, 3, 4, 5, 7, 8, 9, 10, 12, 13, 14, 15>(P, total, st, at)) fold();
  } else {
    bool done = codelets<S, 8, 9, 10, 12, 13, 14, 15>(P, total, st, at);
    if constexpr (HB >= 16)
      if (!done) done = codelets<S, 18, 20, 22, 24, 25, 27, 28, 30, 32, 33>(P, total, st, at);
    if constexpr (HB >= 24)
      if (!done) done = codelets<S, 35, 39, 40, 42, 44, 45, 48, 49>(P, total, st, at);
    if constexpr (HB >= 32)
      if (!done) done = codelets<S, 50, 52, 54, 55, 60, 63, 64, 65>(P, total, st, at);
    if constexpr (FOLD)
      if (!done && A > 1) {
        fold();
        done = true;
      }
    if (!done)
      block_lines<HB, S>(total, st, P, nin, nout, tab, at,
                         [&](At const &z, int q, float2 v) { z.p[q * st] = v; });
  }
#pragma unroll
  for (int e = 0; e < AGD_MAXSP; ++e)
    if (e == d) g.ext[e] = nout;
}

// the window's traces of the nk planes, between LDS and the tiles of U / V
// ([tile of 16 traces][Ft][16] per time window, the last tile as wide as its
// traces): a tile's nk planes are contiguous. Indices by reciprocals (an integer division is ~35
// instructions, and these two loops were most of the kernel's).
// PART: the last tile is narrower (k = rem m / 2^16 divides its rows: rem <
// 4096 and widths up to 16). Windows of 17 x 23 and 16 x 24 traces: 944 and
// 477 us an iteration, 934 and 470 with last tiles padded to 16; as two loops
// 1036 and 531.
template <bool TO_LDS, bool PART>
__device__ __forceinline__ void tiles_loop(float2 *sm, Planes const &g, int ntr, int Ft,
                                           float2 *utw, int k0, int nk) {
  constexpr int NB = 8;  // loads issued together
  int const full = ntr >> 4, wl = ntr & 15;  // whole tiles, width of the last
  int const span = nk * 16, total = nk * ntr;
  unsigned const ml = PART ? 65535u / (unsigned)wl + 1u : 0u, Ft16 = (unsigned)Ft * 16u;
  float const is = 1.f / (float)span;
  float const i1 = 1.f / (float)g.W.y, i2 = 1.f / (float)g.W.z, i3 = 1.f / (float)g.W.w;
  for (int i0 = threadIdx.x; i0 < total; i0 += NB * 256) {
    float2 v[NB];
    int lp[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      int const i = min(i0 + b * 256, total - 1);
      int const t = quot(i, is), rem = i - t * span;
      bool const last = PART && t >= full;
      int const wt = last ? wl : 16;
      int const k = PART ? (int)(__umul24(rem, last ? ml : 4096u) >> 16) : rem >> 4;
      int r = t * 16 + rem - __mul24(k, wt), off = k * g.rp;
      float2 *const u = utw + (__umul24(t, Ft16) + __umul24(k0, wt) + (unsigned)rem);
      if (g.nsp > 3) {
        int const q = quot(r, i3);
        off += (r - q * g.W.w) * g.str.w;
        r = q;
      }
      if (g.nsp > 2) {
        int const q = quot(r, i2);
        off += (r - q * g.W.z) * g.str.z;
        r = q;
      }
      if (g.nsp > 1) {
        int const q = quot(r, i1);
        off += (r - q * g.W.y) * g.str.y;
        r = q;
      }
      off += r * g.str.x;
      lp[b] = i0 + b * 256 < total ? off : -1;
      if (TO_LDS)
        v[b] = *u;
      else if (lp[b] >= 0)
        *u = sm[off];
    }
    if (TO_LDS) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (lp[b] >= 0) sm[lp[b]] = v[b];
    }
  }
}
template <bool TO_LDS>
__device__ __forceinline__ void tiles_copy(float2 *sm, Planes const &g, int ntr, int Ft,
                                           float2 *utw, int k0, int nk) {
  if (ntr & 15)
    tiles_loop<TO_LDS, true>(sm, g, ntr, Ft, utw, k0, nk);
  else
    tiles_loop<TO_LDS, false>(sm, g, ntr, Ft, utw, k0, nk);
}

// mode -1: forward only (X -> U); 0..5 as k_adj_spatial_t's MODE, followed by
// the forward transform of the new model when fuse is set
// FOLD: lines that have two factors fold (HB = 0: all that one FFT does not
// hold; HB = 16: those beyond its codelets, beside lengths that do not fold)
template <int HB, bool FOLD>
__global__ __launch_bounds__(
    256, HB == 0 ? 5 : HB <= 16 ? 4 : HB <= 24 ? 3 : HB <= 32 ? 2 : 1) void k_spatial_g(
    AgdWin const *__restrict__ wins, AgdTask const *__restrict__ tasks, int task0,
    float const *__restrict__ dft, AgdFftPlan const *__restrict__ plans,
    float2 const *__restrict__ roots, float2 const *__restrict__ V, float2 *__restrict__ X,
    float2 *__restrict__ U, float alpha, float lamb, float const *__restrict__ lamb_dev, int mode,
    int fuse, unsigned int *__restrict__ maxbits) {
  extern __shared__ float2 sm[];
  if (lamb_dev != nullptr) lamb = lamb_dev[0];
  AgdTask const t = tasks[task0 + blockIdx.x];
  AgdWin const &w = wins[t.win];
  int const nk = t.nk, nsp = w.nsp, last = w.P[nsp - 1];
  Planes g;
  g.nsp = nsp;
  g.rows = w.S / last;
  g.pitch = last | 1;
  g.rp = g.rows * g.pitch;
  {
    int st = 1;
#pragma unroll
    for (int e = AGD_MAXSP - 1; e >= 0; --e) {
      if (e < nsp) {
        g.P[e] = w.P[e];
        g.W[e] = w.W[e];
        g.A[e] = w.sfac[e];
        g.str[e] = st;
        st *= e == nsp - 1 ? g.pitch : w.P[e];
      } else {
        g.P[e] = g.W[e] = g.str[e] = g.A[e] = 1;
      }
    }
  }
  int64_t const uoff = w.u_off + t.tw * (int64_t)w.uplane;
  float2 *const x = X + w.x_off + ((int64_t)t.tw * w.Ft + t.k0) * w.S;
  int const total = nk * w.S;
  // FOLD: the dims' roots [P_0] .. [P_{n-1}] after the planes (the longest
  // task's: a class's LDS is its largest)
  float2 *const rts = sm + nk * g.rp;
  if constexpr (FOLD) {
    int o = 0;
    for (int d = 0; d < nsp; ++d) {
      int const P = w.P[d];
      for (int m = threadIdx.x; m < P; m += 256) rts[o + m] = roots[plans[w.splan[d]].roots_off + m];
      o += P;
    }
    __syncthreads();
  }
  auto const rt = [&](int d) {
    int o = 0;
#pragma unroll
    for (int e = 0; e < AGD_MAXSP; ++e)
      if (e < d) o += g.P[e];
    return rts + o;
  };
  bool const has_x = mode == -1 || mode == 0 || mode == 2;
  if (mode >= 0) {
#pragma unroll
    for (int e = 0; e < AGD_MAXSP; ++e) g.ext[e] = g.W[e];
    tiles_copy<true>(sm, g, w.ntr, w.Ft, const_cast<float2 *>(V) + uoff, t.k0, nk);
    __syncthreads();
    for (int d = nsp - 1; d >= 0; --d)
      lines<HB, FOLD, -1>(sm, g, nk, d, pick(g.W, d), pick(g.P, d), uniform(dft, w.sdft[d]), rt(d));
  }
  // value i sits at LDS offset i + (row of i) (pitch - last)
  {
    int const pad = g.pitch - last;
    int const dr = 256 / last, dc = 256 - dr * last;
    int row = threadIdx.x / last, col = threadIdx.x - row * last;
    float mx = 0.f;
    constexpr int NB = 8;  // loads issued together
    for (int i0 = threadIdx.x; i0 < total; i0 += NB * 256) {
    float2 v[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (has_x) v[b] = x[min(i0 + b * 256, total - 1)];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      int const i = i0 + b * 256;
      if (i < total) {
        float2 *const s = sm + i + row * pad;
        float2 nv;
        if (mode == -1) {
          nv = v[b];
        } else {
          float2 const gv = *s;
          if (mode == 3) {
            nv = gv;
          } else if (mode == 1 || mode == 4) {
            nv = make_float2(0.f - alpha * gv.x, 0.f - alpha * gv.y);
            float const q = nv.x * nv.x + nv.y * nv.y;
            mx = mode == 1 ? fmaxf(mx, q) : max_bits(mx, q);
          } else {
            nv = step(mode == 5 ? make_float2(0.f, 0.f) : v[b], alpha, gv);
            if (mode == 0 || mode == 5) nv = soft(nv, lamb);
          }
          if (mode != 4) x[i] = nv;
        }
        if (mode == -1 || fuse) *s = nv;
      }
      row += dr;
      col += dc;
      if (col >= last) {
        col -= last;
        ++row;
      }
    }
    }
    if (mode == 1 || mode == 4) {
      __shared__ float red[4];
      for (int o = 32; o > 0; o >>= 1) {
        float const q = __shfl_xor(mx, o, 64);
        mx = mode == 1 ? fmaxf(mx, q) : max_bits(mx, q);
      }
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
      __syncthreads();
      if (threadIdx.x == 0) {
        float m = red[0];
        for (int q = 1; q < 4; ++q) m = mode == 1 ? fmaxf(m, red[q]) : max_bits(m, red[q]);
        atomicMax(maxbits, __float_as_uint(m));
      }
    }
  }
  if (mode == -1 || fuse) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < AGD_MAXSP; ++e) g.ext[e] = g.P[e];
    for (int d = 0; d < nsp; ++d)
      lines<HB, FOLD, +1>(sm, g, nk, d, pick(g.P, d), pick(g.W, d), uniform(dft, w.sdft[d]), rt(d));
    tiles_copy<false>(sm, g, w.ntr, w.Ft, U + uoff, t.k0, nk);
  }
}

// ---------------------------------------------------------------------------
// Time transforms of any even window length, as the complex transform of
// pairs of neighbouring traces, z = x_a + i x_b: no unpack twiddles, and odd
// Pt costs the same as even. A block takes a tile of 16 traces (8 pairs) and
// its time windows [tw0, tw1) as the specialised kernels do; per time window
// the phases run in place on one LDS tile [8][pitch], pitch = 4 mod 8 (lanes
// are (pair, line): the eight pairs start 4 values apart modulo 32, so that a
// phase's reads are free of bank conflicts at an odd line stride).
//
// HB = 0: Pt = M1 M2 M3 with factors up to 16 (M3 = 1: two phases), each
// phase a register FFT. HB > 0: Pt = M1 M2, lines of up to 2 HB + 1 values,
// for the lengths with other primes. Output n = n1 + M1 (n2 + M2 n3) sits at
// n1 M2 M3 + n2 M3 + n3 (pos).
//
// Latency bounds these kernels (loads, barriers, a phase's few lines), and
// waves hide it, so short factors pay twice: fewer instructions, and
// registers for more waves. Measured on the volume above (Pt = 250 = 10 x 5 x
// 5, 1.0 GB a launch), forward and adjoint: lines of 10 x 25 484 and 500 us
// (four waves to a SIMD, 220 million vector instructions), now 291 and 278
// (six, 129 million). A register prefetch of the next tile in the forward,
// which takes waves, ran 656 against 484 us.
// ---------------------------------------------------------------------------
constexpr int kPairs = 8;
__host__ __device__ constexpr int time_pitch(int Pt) { return (Pt + 3) / 8 * 8 + 4; }

// rows of a tile are as wide as its nt traces: the pair p of row k starts at
// value k nt + 2 p, which item i = k np + p (np pairs a row, the last of an odd
// nt a single) finds at 2 i - (nt odd ? k : 0). 16 bytes aligned to 8.
typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));

struct TimeTables {
  float2 *Z, *TW, *TW2;
  unsigned short *pos;
};

template <int S>
__device__ __forceinline__ void time_tables(TimeTables const &t, float2 const *roots, int N,
                                            int M1, int M2, int M3) {
  float const i1 = 1.f / (float)M1, i2 = 1.f / (float)M2;
  for (int m = threadIdx.x; m < N; m += 256) {
    // TW[r M1 + n1] = exp(S 2 pi i n1 r / N)
    int const r = quot(m, i1), n1 = m - r * M1, n3 = quot(r, i2), n2 = r - n3 * M2;
    float2 const z = roots[n1 * r];  // n1 r < N
    t.TW[m] = make_float2(z.x, S > 0 ? -z.y : z.y);
    t.pos[m] = (unsigned short)((n1 * M2 + n2) * M3 + n3);
    // TW2[k3 M2 + n2] = exp(S 2 pi i n2 k3 / (M2 M3))
    if (M3 > 1 && n1 == 0) {
      float2 const y = roots[n2 * n3 * M1];
      t.TW2[r] = make_float2(y.x, S > 0 ? -y.y : y.y);
    }
  }
}

// a phase's lines as register FFTs of a length in Ps: line l of at(l), stride
// st, output q through put(line, q, st, value). (st passes through an empty
// asm, so that the sums of the addresses are not kept, in registers that then
// spilled, beyond their use.)
template <int S, class At, class Put>
__device__ __forceinline__ void phase(int, int, int, At const &, Put const &) {}
template <int S, int N, int... Ps, class At, class Put>
__device__ __forceinline__ void phase(int P, int total, int st, At const &at, Put const &put) {
  if (P != N) {
    phase<S, Ps...>(P, total, st, at, put);
    return;
  }
  int l = threadIdx.x;
  asm volatile("" : "+v"(l), "+s"(st));
  for (; l < total; l += 256) {
    auto const z = at(l);
    float2 v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = z.p[k * st];
    agdfft::fft<N, S>(v);
    asm volatile("" : "+s"(st) : : "memory");
#pragma unroll
    for (int k = 0; k < N; ++k) put(z, k, st, v[k]);
  }
}

template <int HB, int S>
__device__ __forceinline__ void time_fft(TimeTables const &t, int pitch, int M1, int M2, int M3,
                                         float const *dft, int d1, int d2) {
  struct At {
    float2 *p;
    float2 const *tw;
  };
  int const M23 = M2 * M3;
  auto const twiddled = [](At const &z, int q, int st, float2 v) {
    z.p[q * st] = q == 0 ? v : agdfft::c_mul(v, z.tw[q]);
  };
  auto const plain = [](At const &z, int q, int st, float2 v) { z.p[q * st] = v; };
  auto const at1 = [&](int l) {
    int const p = l % kPairs, r = l / kPairs;
    return At{t.Z + p * pitch + r, t.TW + r * M1};
  };
  auto const at2 = [&](int l) {  // M3 = 1
    int const p = l % kPairs, n1 = l / kPairs;
    return At{t.Z + p * pitch + n1 * M2, nullptr};
  };
  auto const run = [&](int P, int total, int st, auto const &at, auto const &put) {
    phase<S, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>(P, total, st, at, put);
    __syncthreads();
  };
  if constexpr (HB == 0) {
    run(M1, kPairs * M23, M23, at1, twiddled);
    if (M3 == 1) {
      run(M2, kPairs * M1, 1, at2, plain);
    } else {
      float const i3 = 1.f / (float)M3;
      run(M2, kPairs * M1 * M3, M3,
          [&](int l) {
            int const p = l % kPairs, r = l / kPairs, n1 = quot(r, i3), k3 = r - n1 * M3;
            return At{t.Z + p * pitch + n1 * M23 + k3, t.TW2 + k3 * M2};
          },
          twiddled);
      run(M3, kPairs * M1 * M2, 1,
          [&](int l) {
            int const p = l % kPairs, r = l / kPairs;
            return At{t.Z + p * pitch + r * M3, nullptr};
          },
          plain);
    }
  } else {
    if (M1 > 1)
      block_lines<HB, S>(kPairs * M2, M2, M1, M1, M1, uniform(dft, d1), at1,
                         [&](At const &z, int q, float2 v) { twiddled(z, q, M2, v); });
    block_lines<HB, S>(kPairs * M1, 1, M2, M2, M2, uniform(dft, d2), at2,
                       [&](At const &z, int q, float2 v) { plain(z, q, 1, v); });
  }
}

// waves per SIMD that the registers are bounded for
constexpr int time_waves(int HB) { return HB == 0 ? 6 : HB <= 16 ? 4 : HB <= 32 ? 2 : 1; }

template <int HB>
__global__ __launch_bounds__(256, time_waves(HB)) void k_fwd_time_g(
    AgdWin const *__restrict__ wins, int const *__restrict__ blocks, int block0,
    float const *__restrict__ dft, AgdFftPlan const *__restrict__ plans,
    float2 const *__restrict__ roots, float const *__restrict__ tapers,
    float const *__restrict__ tscale, float2 const *__restrict__ U, float *__restrict__ T) {
  extern __shared__ float2 sm[];
  int const *const bl = blocks + TB_INTS * (block0 + blockIdx.x);
  AgdWin const &w = wins[bl[0]];
  int const t0 = bl[1], nt = min(2 * kPairs, w.ntr - t0);
  int const twn = bl[3] - bl[2];
  int const tw0 = bl[2] + twn * blockIdx.y / gridDim.y;
  int const tw1 = bl[2] + twn * (blockIdx.y + 1) / gridDim.y;
  int const twa = tw0 > 0 ? tw0 - 1 : 0;
  int const N = w.Pt, Ft = w.Ft, Wt = w.Wt, half = w.half, M1 = w.gm1, M2 = w.gm2, M3 = max(w.gm3, 1);
  int const nconv = w.nconv, ntw = w.ntw, pitch = time_pitch(N);
  TimeTables t;
  t.Z = sm;
  t.TW = t.Z + kPairs * pitch;
  t.TW2 = t.TW + N;  // [M2 M3], unless M3 = 1
  float *const TP = (float *)(t.TW2 + (M3 > 1 ? M2 * M3 : 0));    // [Wt] time taper
  float *const CA = TP + Wt;                // [16][half] overlap carry
  t.pos = (unsigned short *)(CA + 2 * kPairs * half);
  int const tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = 4;
  time_tables<+1>(t, roots + plans[w.tplan_full].roots_off, N, M1, M2, M3);
  for (int i = tid; i < Wt; i += 256) TP[i] = tapers[w.tt_off + i];
  for (int i = tid; i < 2 * kPairs * half; i += 256) CA[i] = 0.f;
  float *const Tb = T + w.t_off + (int64_t)t0 * nconv;
  float2 const *const tile = U + w.u_off + (int64_t)t0 * Ft;
  int const np = (nt + 1) >> 1, odd = nt & 1;
  float const ip = 1.f / (float)np;
  for (int tw = twa; tw < tw1; ++tw) {
    float2 const *const u = tile + tw * (int64_t)w.uplane;
    // Hermitian halves of both traces of a pair into z = x_a + i x_b (DC and
    // Nyquist imaginary parts ignored). A single's partner is zero: its load
    // takes the next row's first value, or the one past the tile (the buffer
    // has one more). Pairs beyond np transform what the tile holds, unused.
    constexpr int NB = 4;
    for (int i0 = tid; i0 < Ft * np; i0 += NB * 256) {
      f4u v[NB];
      int kk[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        int const i = min(i0 + b * 256, Ft * np - 1);
        kk[b] = quot(i, ip);
        v[b] = *(f4u const *)(u + 2 * i - (odd ? kk[b] : 0));
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        int const i = i0 + b * 256;
        if (i < Ft * np) {
          int const k = kk[b], p = i - k * np;
          float2 xa = make_float2(v[b].x, v[b].y), xb = make_float2(v[b].z, v[b].w);
          if (2 * p + 1 >= nt) xb = make_float2(0.f, 0.f);
          if (k == 0 || 2 * k == N) xa.y = xb.y = 0.f;
          float2 *const z = t.Z + p * pitch;
          z[k] = make_float2(xa.x - xb.y, xa.y + xb.x);
          if (k > 0 && 2 * k < N) z[N - k] = make_float2(xa.x + xb.y, xb.x - xa.y);
        }
      }
    }
    __syncthreads();
    time_fft<HB, +1>(t, pitch, M1, M2, M3, dft, w.tdft1, w.tdft2);
    // overlap-add: samples [0, half) complete this window's first half
    for (int p = wave; p < kPairs; p += nw) {
      if (2 * p >= nt) break;
      float const sa = tscale[w.trace0 + t0 + 2 * p];
      float const sb = tscale[w.trace0 + t0 + min(2 * p + 1, nt - 1)];
      float2 const *const z = t.Z + p * pitch;
      float *const ca = CA + 2 * p * half, *const cb = ca + half;
      float *const ta = Tb + (int64_t)2 * p * nconv + tw * half, *const tb = ta + nconv;
      for (int s = lane; s < half; s += 64) {
        float2 const z0 = z[t.pos[s]], z1 = z[t.pos[s + half]];
        float const w0 = TP[s], w1 = TP[s + half];
        if (tw >= tw0) {
          ta[s] = ca[s] + z0.x * sa * w0;
          if (2 * p + 1 < nt) tb[s] = cb[s] + z0.y * sb * w0;
        }
        ca[s] = z1.x * sa * w1;
        cb[s] = z1.y * sb * w1;
      }
    }
    __syncthreads();
  }
  if (tw1 < ntw) return;
  for (int j = wave; j < nt; j += nw) {
    float *const tj = Tb + (int64_t)j * nconv;
    for (int s = lane; s < half; s += 64)
      if (ntw * half + s < nconv) tj[ntw * half + s] = CA[j * half + s];
  }
}

template <int HB>
__global__ __launch_bounds__(256, time_waves(HB)) void k_adj_time_g(
    AgdWin const *__restrict__ wins, int const *__restrict__ blocks, int block0,
    float const *__restrict__ dft, AgdFftPlan const *__restrict__ plans,
    float2 const *__restrict__ roots, float const *__restrict__ tapers,
    float const *__restrict__ tscale, AgdEntry const *__restrict__ went,
    float const *__restrict__ rec, float const *__restrict__ Tin, float2 *__restrict__ V,
    int plain, int const *__restrict__ order) {
  extern __shared__ float2 sm[];
  // the launch order of the specialised kernel (neighbouring windows' blocks
  // of the same traces on one XCD)
  int const bid = order ? order[block0 + xcd_chunk(blockIdx.x, gridDim.x)] : block0 + blockIdx.x;
  int const *const bl = blocks + TB_INTS * bid;
  AgdWin const &w = wins[bl[0]];
  int const t0 = bl[1], nt = min(2 * kPairs, w.ntr - t0);
  int const twn = bl[3] - bl[2];
  int const tw0 = bl[2] + twn * blockIdx.y / gridDim.y;
  int const tw1 = bl[2] + twn * (blockIdx.y + 1) / gridDim.y;
  int const N = w.Pt, Ft = w.Ft, Wt = w.Wt, half = w.half, M1 = w.gm1, M2 = w.gm2, M3 = max(w.gm3, 1);
  int const nconv = w.nconv, pitch = time_pitch(N);
  TimeTables t;
  t.Z = sm;
  t.TW = t.Z + kPairs * pitch;
  t.TW2 = t.TW + N;  // [M2 M3], unless M3 = 1
  float *const TP = (float *)(t.TW2 + (M3 > 1 ? M2 * M3 : 0));
  t.pos = (unsigned short *)(TP + Wt);
  int const tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  time_tables<-1>(t, roots + plans[w.tplan_full].roots_off, N, M1, M2, M3);
  for (int i = tid; i < Wt; i += 256) TP[i] = plain ? 1.f : tapers[w.tt_off + i];
  __syncthreads();
  // one source: the record through the blend entries, or a trace buffer; a
  // wave takes two pairs of traces, whose entries and scales stay in registers
  float const *const src = Tin != nullptr ? Tin : rec;
  constexpr int NP = kPairs / 4;
  int64_t at[NP][2];
  int start[NP][2], cnt[NP][2];
  float sc[NP][2];
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      int const j = 2 * (wave + 4 * i) + q, jc = min(j, nt - 1);
      AgdEntry const e = went[w.trace0 + t0 + jc];
      float const ts = tscale[w.trace0 + t0 + jc];
      at[i][q] = Tin != nullptr ? w.t_off + (int64_t)(t0 + jc) * nconv : e.rec;
      start[i][q] = Tin != nullptr ? 0 : e.trace_start;
      cnt[i][q] = j >= nt ? 0 : Tin != nullptr ? nconv : e.n;
      sc[i][q] = plain ? w.scaler : ts;
    }
  // unconditional loads (index clamped into the trace's range), zeroed
  // outside it, so that they stay in flight together
  auto sample = [&](int i, int q, int t, bool in) -> float {
    int const i2 = t - start[i][q];
    bool const ok = in && (unsigned)i2 < (unsigned)cnt[i][q];
    float const v = src[at[i][q] + (ok ? i2 : 0)];
    return ok ? v : 0.f;
  };
  float const two = plain ? 1.f : 2.f;
  int const kmax2 = (N - 1) / 2;
  float2 *const vt = V + w.u_off + (int64_t)t0 * Ft;
  int const np = (nt + 1) >> 1, odd = nt & 1;
  float const ip = 1.f / (float)np;
  for (int tw = tw0; tw < tw1; ++tw) {
    constexpr int NB = 2;
    for (int s0 = lane; s0 < N; s0 += 64 * NB) {
      float x[NP][NB][2];
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            int const s = s0 + 64 * b;
            x[i][b][q] = sample(i, q, tw * half + s, s < Wt);
          }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        int const s = s0 + 64 * b;
        float const tp = TP[min(s, Wt - 1)];
        if (s < N) {
#pragma unroll
          for (int i = 0; i < NP; ++i)
            t.Z[(wave + 4 * i) * pitch + s] =
                make_float2(x[i][b][0] * sc[i][0] * tp, x[i][b][1] * sc[i][1] * tp);
        }
      }
    }
    __syncthreads();
    time_fft<HB, -1>(t, pitch, M1, M2, M3, dft, w.tdft1, w.tdft2);
    // half spectra of the two real traces of a pair, x2 on the interior bins
    float2 *const vo = vt + tw * (int64_t)w.uplane;
    for (int i = tid; i < Ft * np; i += 256) {
      int const k = quot(i, ip), p = i - k * np;
      float2 const *const z = t.Z + p * pitch;
      float2 const z1 = z[t.pos[k]], z2 = z[t.pos[k ? N - k : 0]];
      float const s = (k >= 1 && k <= kmax2) ? 0.5f * two : 0.5f;
      float2 *const o = vo + 2 * i - (odd ? k : 0);
      float2 const va = make_float2(s * (z1.x + z2.x), s * (z1.y - z2.y));
      if (2 * p + 1 < nt)
        *(f4u *)o = f4u{va.x, va.y, s * (z1.y + z2.y), s * (z2.x - z1.x)};
      else
        *o = va;
    }
    __syncthreads();
  }
}

// Instances of the run-time sized kernels by the coefficient pairs HB a line
// holds in registers (lengths up to 2 HB + 1): the fewer, the more waves
// share a SIMD. The host picks the smallest that fits a window's lines.
template <int HB, bool FOLD>
static int launch_spatial_g(AgdDev const *g, AgdClass const &c, float2 *X, float alpha,
                            float lamb, int mode, int fuse) {
  static int const lds_ok = allow_lds((void const *)k_spatial_g<HB, FOLD>);
  (void)lds_ok;
  int first;
  int const n = class_range(g, c, &first);
  if (n <= 0) return 0;
  return launch(mode < 0 ? "fwd_spatial" : "adj_spatial", k_spatial_g<HB, FOLD>, dim3(n),
                dim3(NTHR), c.lds, g->win, g->tasks, first, g->dft, g->plans,
                (float2 const *)g->roots, (float2 const *)g->V, X,
                (float2 *)g->U, alpha, lamb, (float const *)g->lamb_dev, mode, fuse, g->scalar);
}
int spatial_general(AgdDev const *g, AgdClass const &c, float2 *X, float alpha,
                           float lamb, int mode, int fuse) {
  switch (c.hb) {
    case AGD_FACTORED: return launch_spatial_g<0, true>(g, c, X, alpha, lamb, mode, fuse);
    case AGD_FOLDED_LINES: return launch_spatial_g<16, true>(g, c, X, alpha, lamb, mode, fuse);
    case 8: return launch_spatial_g<8, false>(g, c, X, alpha, lamb, mode, fuse);
    case 16: return launch_spatial_g<16, false>(g, c, X, alpha, lamb, mode, fuse);
    case 24: return launch_spatial_g<24, false>(g, c, X, alpha, lamb, mode, fuse);
    case 32: return launch_spatial_g<32, false>(g, c, X, alpha, lamb, mode, fuse);
    case 48: return launch_spatial_g<48, false>(g, c, X, alpha, lamb, mode, fuse);
    default: return launch_spatial_g<64, false>(g, c, X, alpha, lamb, mode, fuse);
  }
}
template <int HB>
static int launch_fwd_time_g(AgdDev const *g, AgdClass const &c, int first, int n) {
  static int const lds_ok = allow_lds((void const *)k_fwd_time_g<HB>);
  (void)lds_ok;
  // by registers, and by the LDS of a CU
  static int const held = agd_resident((void const *)k_fwd_time_g<HB>, NTHR, 0);
  int const fits = agd_compute_units() * (int)(160 * 1024 / c.lds);
  int const runs = time_split_fwd(g, c, n, held < fits ? held : fits);
  return launch("fwd_time", k_fwd_time_g<HB>, dim3(n, runs), dim3(NTHR), c.lds, g->win,
                g->tblocks, first, g->dft, g->plans, (float2 const *)g->roots, g->tapers,
                g->tscale, (float2 const *)g->U, g->T);
}
int fwd_time_general(AgdDev const *g, AgdClass const &c, int first, int n) {
  switch (c.hb) {
    case AGD_FACTORED: return launch_fwd_time_g<0>(g, c, first, n);
    case 8: return launch_fwd_time_g<8>(g, c, first, n);
    case 16: return launch_fwd_time_g<16>(g, c, first, n);
    case 32: return launch_fwd_time_g<32>(g, c, first, n);
    default: return launch_fwd_time_g<64>(g, c, first, n);
  }
}
template <int HB>
static int launch_adj_time_g(AgdDev const *g, AgdClass const &c, int first, int n,
                             float const *Tin, int plain) {
  static int const lds_ok = allow_lds((void const *)k_adj_time_g<HB>);
  (void)lds_ok;
  return launch("adj_time", k_adj_time_g<HB>, dim3(n, time_split(g, c, n, 1)), dim3(NTHR), c.lds, g->win,
                g->tblocks, first, g->dft, g->plans, (float2 const *)g->roots, g->tapers,
                g->tscale, g->went, (float const *)g->r, Tin, (float2 *)g->V, plain,
                first == c.begin && n == c.count ? g->tadj : (int const *)nullptr);
}
int adj_time_general(AgdDev const *g, AgdClass const &c, int first, int n,
                            float const *Tin, int plain) {
  switch (c.hb) {
    case AGD_FACTORED: return launch_adj_time_g<0>(g, c, first, n, Tin, plain);
    case 8: return launch_adj_time_g<8>(g, c, first, n, Tin, plain);
    case 16: return launch_adj_time_g<16>(g, c, first, n, Tin, plain);
    case 32: return launch_adj_time_g<32>(g, c, first, n, Tin, plain);
    default: return launch_adj_time_g<64>(g, c, first, n, Tin, plain);
  }
}

}  // namespace agdgen
