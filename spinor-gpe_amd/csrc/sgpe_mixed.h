// Split-step passes and standalone transforms for even lengths without a
// compiled power-of-two kernel whose prime factors are at most 13, 32 to 2048
// points. An inner stage has one butterfly per thread and a workgroup 512 threads:
// columns and transforms of 1694, 1716, 1782, 2002 and 2028 points and rows (two
// components at a time) of those and 1452, 1458, 1750, 1848, 1936, 1944 and 1980
// have more and stay with sgpe_generic.h, as all other lengths do.
//
// A length is split on the host into two to four radices of at most 16
// (mix_factor). A stage is one register butterfly of compile-time radix per
// work item (a uniform switch picks the radix); data pass between stages through
// LDS. A pass runs
//     stage 0 (global -> LDS), inner stages (LDS -> LDS), last stage,
//     pointwise block, then the adjoint stages back in reverse order:
// the second transform is the conjugate transpose of the first, stage by
// stage, so it reads the same twiddle table, its first stage works on the very
// points a thread holds after the last stage of the first transform (in place in
// LDS; the column pass applies its factors between the two in registers), and
// its last stage writes to global memory what stage 0 read. Against keeping the
// data in LDS throughout, with one stage per prime power, twiddles gathered from
// global memory and two LDS buffers (sgpe_generic.h), a 600-point column
// pass makes 4 round trips through LDS instead of 10 (the row pass 6).
//
// Bound by latency on grids of this size (one or two workgroups per CU: each
// stage is an LDS round trip and a barrier), by LDS and vector instructions in
// batches. Measured (dispatch times, us, sgpe_generic.h -> here): 600 x 480
// complex128 column 30.9 -> 18.5, row 23.8 -> 15.6; 1000^2 complex64 column 52.1
// -> 22.2, row 34.7 -> 21.7; 1536^2 complex128 column 168 -> 67, row 190 -> 92.
#pragma once

#include <type_traits>

#include "sgpe_kernels.h"
#include "sgpe_units.h"

namespace sgpe {

constexpr int kMixMaxStages = 4;
constexpr int kMixMaxLen = 2048;
constexpr int kMixMinLen = 32;
constexpr int kMixMaxRadix = 16;
constexpr int kMixMidRadix = 10;  // last stage: holds its twiddles
constexpr int kMixThreads = 512;  // most threads of a workgroup

// One stage: radix, span (product of the radices before it), butterflies,
// offset of its twiddles, and multipliers for exact division of 16-bit numbers
// by span and butterflies (floor(2^32 / d) + 1).
struct MixStage {
  int radix, span, nb, off;
  unsigned div_span, div_nb;
};
struct MixFft {
  int n, ns;
  MixStage st[kMixMaxStages];
};

// x / d for x, d < 2^16 with m = floor(2^32 / d) + 1 (d = 1: m wraps to 1;
// answered apart).
__device__ __forceinline__ int mix_div(int x, int d, unsigned m) {
  return d == 1 ? x : (int)__umulhi((unsigned)x, m);
}

// ------------------------------------------------------ register butterflies

// Odd prime radix: sums and differences of opposite inputs. From radix 7 on the
// products and sums run in double also for complex64 (the same instruction
// rate): the rounded constants of a float DFT_13 repeat in every pass, so their
// errors add up coherently (10 real-time steps of 286^2: 2.4e-6 relative error
// instead of 1.9e-6).
template <int R, bool INV, typename C> __device__ __forceinline__ void dft_odd(C (&b)[R]) {
  typedef decltype(b[0].x) S;
  typedef typename std::conditional<(R >= 7), double, S>::type A;
  constexpr int H = (R - 1) / 2;
  A tx[H], ty[H], dx[H], dy[H];
  const A bx = (A)b[0].x, by = (A)b[0].y;
  A yx = bx, yy = by;
#pragma unroll
  for (int j = 0; j < H; ++j) {
    const A px = (A)b[j + 1].x, py = (A)b[j + 1].y, qx = (A)b[R - 1 - j].x, qy = (A)b[R - 1 - j].y;
    tx[j] = px + qx;
    ty[j] = py + qy;
    dx[j] = px - qx;
    dy[j] = py - qy;
    yx += tx[j];
    yy += ty[j];
  }
  b[0] = C{(S)yx, (S)yy};
#pragma unroll
  for (int q = 1; q <= H; ++q) {
    A ax = bx, ay = by, sx = 0, sy = 0;
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const A cj = (A)MixUnitTable<R>::u.c[((j + 1) * q) % R], sj = (A)MixUnitTable<R>::u.s[((j + 1) * q) % R];
      ax += cj * tx[j];
      ay += cj * ty[j];
      sx += sj * dx[j];
      sy += sj * dy[j];
    }
    const C lo = C{(S)(ax + sy), (S)(ay - sx)}, hi = C{(S)(ax - sy), (S)(ay + sx)};
    b[q] = INV ? hi : lo;
    b[R - q] = INV ? lo : hi;
  }
}

template <int R, bool INV, typename C> __device__ __forceinline__ void mix_dft(C (&b)[R]);

// R = R1 R2 with coprime factors: no twiddles between the two levels (input
// index (R2 n1 + R1 n2) mod R, output index k = k1 mod R1 = k2 mod R2).
template <int R1, int R2, bool INV, typename C> __device__ __forceinline__ void dft_coprime(C (&b)[R1 * R2]) {
  constexpr int R = R1 * R2;
  C x[R];
#pragma unroll
  for (int n2 = 0; n2 < R2; ++n2) {
    C u[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) u[n1] = b[(R2 * n1 + R1 * n2) % R];
    mix_dft<R1, INV>(u);
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) x[k1 * R2 + n2] = u[k1];
  }
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) {
    C u[R2];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) u[n2] = x[k1 * R2 + n2];
    mix_dft<R2, INV>(u);
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k % R1 == k1) b[k] = u[k % R2];
  }
}

template <bool INV, typename C> __device__ __forceinline__ void dft9(C (&b)[9]) {
  typedef decltype(b[0].x) S;
  C x[9];
#pragma unroll
  for (int n2 = 0; n2 < 3; ++n2) {
    C u[3] = {b[n2], b[3 + n2], b[6 + n2]};
    dft_odd<3, INV>(u);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      // Constants in double for the same reason as in dft_odd.
      const double c = MixUnitTable<9>::u.c[n2 * k1], s = (INV ? 1.0 : -1.0) * MixUnitTable<9>::u.s[n2 * k1];
      const double ux = u[k1].x, uy = u[k1].y;
      x[k1 * 3 + n2] = n2 * k1 ? C{(S)(ux * c - uy * s), (S)(ux * s + uy * c)} : u[k1];
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    C u[3] = {x[k1 * 3], x[k1 * 3 + 1], x[k1 * 3 + 2]};
    dft_odd<3, INV>(u);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) b[k1 + 3 * k2] = u[k2];
  }
}

// Natural-order DFT of R points in registers.
template <int R, bool INV, typename C> __device__ __forceinline__ void mix_dft(C (&b)[R]) {
  if constexpr (R == 2 || R == 4 || R == 8 || R == 16)
    dft<R, INV>(b);
  else if constexpr (R == 6)
    dft_coprime<2, 3, INV>(b);
  else if constexpr (R == 9)
    dft9<INV>(b);
  else if constexpr (R == 10)
    dft_coprime<2, 5, INV>(b);
  else if constexpr (R == 12)
    dft_coprime<4, 3, INV>(b);
  else if constexpr (R == 14)
    dft_coprime<2, 7, INV>(b);
  else if constexpr (R == 15)
    dft_coprime<3, 5, INV>(b);
  else
    dft_odd<R, INV>(b);
}

// f(PointVariant<R>) for a stage's radix (uniform). MAXR: largest compiled.
template <int MAXR, class F> __device__ __forceinline__ void mix_radix(int radix, F&& f) {
#define SGPE_MIX_CASE(R) \
  case R:                \
    if constexpr (R <= MAXR) f(PointVariant<R>()); \
    break;
  switch (radix) {
    SGPE_MIX_CASE(2) SGPE_MIX_CASE(3) SGPE_MIX_CASE(4) SGPE_MIX_CASE(5) SGPE_MIX_CASE(6) SGPE_MIX_CASE(7)
    SGPE_MIX_CASE(8) SGPE_MIX_CASE(9) SGPE_MIX_CASE(10) SGPE_MIX_CASE(11) SGPE_MIX_CASE(12) SGPE_MIX_CASE(13)
    SGPE_MIX_CASE(14) SGPE_MIX_CASE(15) SGPE_MIX_CASE(16)
    default: break;
  }
#undef SGPE_MIX_CASE
}

// The transforms of one workgroup in LDS: `batch` of them, element i of
// transform m at base[m * ms + i * is]. Work item w of a stage is butterfly v
// of transform m; columns (is > 1) take neighbouring transforms in
// neighbouring items, rows (is = 1) neighbouring butterflies.
template <typename C> struct MixTile {
  C* lds;
  const C* tw;
  int batch, ms, is;
  unsigned div_batch;
  __device__ __forceinline__ void item(const MixStage& st, int w, int* m, int* v) const {
    if (is == 1) {
      *m = mix_div(w, st.nb, st.div_nb);
      *v = w - *m * st.nb;
    } else {
      *v = mix_div(w, batch, div_batch);
      *m = w - *v * batch;
    }
  }
  __device__ __forceinline__ C& at(int m, int i) const { return lds[m * ms + i * is]; }
};

// Twiddles of butterfly position k of a stage, conjugated for the inverse.
template <int R, bool INV, typename C>
__device__ __forceinline__ void mix_twiddle(C (&b)[R], const C* __restrict__ w) {
#pragma unroll
  for (int r = 1; r < R; ++r) {
    C t = w[r - 1];
    if (INV) t.y = -t.y;
    b[r] = cmul(b[r], t);
  }
}

// Stage 0 of the first transform: butterflies of elements read with
// rd(m, i), written to LDS. No barrier.
template <bool INV, typename C, class Rd>
__device__ __forceinline__ void mix_first(const MixFft& f, const MixTile<C>& x, Rd rd) {
  const MixStage& st = f.st[0];
  const int items = st.nb * x.batch;
  mix_radix<kMixMaxRadix>(st.radix, [&](auto rr) {
    constexpr int R = decltype(rr)::v;
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
      int m, v;
      x.item(st, w, &m, &v);
      C b[R];
#pragma unroll
      for (int r = 0; r < R; ++r) b[r] = rd(m, v + r * st.nb);
      mix_dft<R, INV>(b);
#pragma unroll
      for (int q = 0; q < R; ++q) x.at(m, v * R + q) = b[q];
    }
  });
}

// Inner stages 1 .. ns - 2 of the first transform, in place in LDS: a work
// item per thread (the host sees to it), a barrier between all reads and all
// writes. Starts and ends with a barrier.
template <bool INV, typename C>
__device__ __forceinline__ void mix_inner(const MixFft& f, const MixTile<C>& x) {
  __syncthreads();
  for (int s = 1; s < f.ns - 1; ++s) {
    const MixStage& st = f.st[s];
    const bool on = (int)threadIdx.x < st.nb * x.batch;
    mix_radix<kMixMaxRadix>(st.radix, [&](auto rr) {
      constexpr int R = decltype(rr)::v;
      int m = 0, v = 0, k = 0;
      C b[R];
      if (on) {
        x.item(st, threadIdx.x, &m, &v);
        k = v - mix_div(v, st.span, st.div_span) * st.span;
#pragma unroll
        for (int r = 0; r < R; ++r) b[r] = x.at(m, v + r * st.nb);
        mix_twiddle<R, INV>(b, x.tw + st.off + k * (R - 1));
        mix_dft<R, INV>(b);
      }
      __syncthreads();
      if (on) {
        const int base = (v - k) * R + k;
#pragma unroll
        for (int q = 0; q < R; ++q) x.at(m, base + q * st.span) = b[q];
      }
    });
    __syncthreads();
  }
}

// Adjoint inner stages ns - 2 .. 1 of the second transform (direction INV).
template <bool INV, typename C>
__device__ __forceinline__ void mix_inner_adj(const MixFft& f, const MixTile<C>& x) {
  __syncthreads();
  for (int s = f.ns - 2; s > 0; --s) {
    const MixStage& st = f.st[s];
    const bool on = (int)threadIdx.x < st.nb * x.batch;
    mix_radix<kMixMaxRadix>(st.radix, [&](auto rr) {
      constexpr int R = decltype(rr)::v;
      int m = 0, v = 0;
      C b[R];
      if (on) {
        x.item(st, threadIdx.x, &m, &v);
        const int k = v - mix_div(v, st.span, st.div_span) * st.span;
        const int base = (v - k) * R + k;
#pragma unroll
        for (int q = 0; q < R; ++q) b[q] = x.at(m, base + q * st.span);
        mix_dft<R, INV>(b);
        mix_twiddle<R, INV>(b, x.tw + st.off + k * (R - 1));
      }
      __syncthreads();
      if (on) {
#pragma unroll
        for (int r = 0; r < R; ++r) x.at(m, v + r * st.nb) = b[r];
      }
    });
    __syncthreads();
  }
}

// Adjoint of stage 0: the last stage of the second transform, elements
// handed to wr(m, i, value).
template <bool INV, typename C, class Wr>
__device__ __forceinline__ void mix_first_adj(const MixFft& f, const MixTile<C>& x, Wr wr) {
  const MixStage& st = f.st[0];
  const int items = st.nb * x.batch;
  mix_radix<kMixMaxRadix>(st.radix, [&](auto rr) {
    constexpr int R = decltype(rr)::v;
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
      int m, v;
      x.item(st, w, &m, &v);
      C b[R];
#pragma unroll
      for (int q = 0; q < R; ++q) b[q] = x.at(m, v * R + q);
      mix_dft<R, INV>(b);
#pragma unroll
      for (int r = 0; r < R; ++r) wr(m, v + r * st.nb, b[r]);
    }
  });
}

// The twiddle table (n - 1 entries) into LDS: load() issues the first four
// loads of a thread ahead of the state's, store() writes them (and the rest).
template <typename C> struct MixTwiddles {
  C v[4];
  __device__ __forceinline__ void load(const C* __restrict__ tw, int n) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = threadIdx.x + k * (int)blockDim.x;
      v[k] = ld_global(tw + (i < n - 1 ? i : 0));
    }
  }
  __device__ __forceinline__ void store(const C* __restrict__ tw, int n, C* dst) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = threadIdx.x + k * (int)blockDim.x;
      if (i < n - 1) dst[i] = v[k];
    }
    for (int i = threadIdx.x + 4 * (int)blockDim.x; i < n - 1; i += blockDim.x) dst[i] = ld_global(tw + i);
  }
};

// ------------------------------------------------------------ column pass
// W columns of component blockIdx.y of slot blockIdx.z, as col_pass_kernel.
// LDS: [n W data][n twiddles][sums].
template <typename R>
__global__ __launch_bounds__(kMixThreads) void mix_col_pass_kernel(const InstDev* __restrict__ insts,
                                                                   RunDev* __restrict__ runs, MixFft f,
                                                                   const typename Cx<R>::T* __restrict__ tw, int W,
                                                                   unsigned div_w, int mode, int d_prev, int d_cur) {
  typedef typename Cx<R>::T C;
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  if (!runs[inst].active) return;
  const InstDev& P = insts[inst];
  const bool kspace = runs[inst].form == FORM_KSPACE;
  const int N = f.n, nx = P.nx, comp = blockIdx.y;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int jx0 = tile * W;
  C* const psi = reinterpret_cast<C*>(P.psi) + (size_t)comp * N * nx + jx0;
  MixTile<C> x;
  x.lds = reinterpret_cast<C*>(smem);
  C* const twl = x.lds + N * W;
  x.tw = twl;
  x.batch = W;
  x.div_batch = div_w;
  x.ms = 1;
  x.is = W;
  MixTwiddles<C> stw;
  stw.load(tw, N);
  if (!kspace) mix_first<false, C>(f, x, [&](int m, int i) { return ld_global(psi + (size_t)i * nx + m); });
  stw.store(tw, N, twl);
  if (!kspace)
    mix_inner<false>(f, x);
  else
    __syncthreads();

  // Last stage, kinetic factors (as col_pass_kernel), adjoint last stage.
  const double* td = P.t_dense[comp];
  const bool mid = mode != COL_EXIT, want_s = mode == COL_MID_S, imag = P.imag != 0;
  const bool one = !imag && (kspace || !mid);
  const int d1 = kspace ? d_cur : d_prev;
  const C* kxt = reinterpret_cast<const C*>(one ? P.kx[d1][comp] : P.k2x[d_prev][d_cur][comp]);
  const C* kyt = reinterpret_cast<const C*>(one ? P.ky[d1][comp] : P.k2y[d_prev][d_cur][comp]);
  const R hp = (R)(0.5 * P.dt_sub[d_prev]), hc = (R)(0.5 * P.dt_sub[d_cur]);
  double s_acc = 0.0, n_acc = 0.0;
  const MixStage& st = f.st[f.ns - 1];
  const int items = st.nb * W;
  mix_radix<kMixMidRadix>(st.radix, [&](auto rr) {
    constexpr int E = decltype(rr)::v;
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
      int m, v;
      x.item(st, w, &m, &v);
      const int jx = jx0 + m;
      const C* wk = x.tw + st.off + v * (E - 1);  // k = v: the span is n / radix
      C b[E];
      if (kspace) {
#pragma unroll
        for (int r = 0; r < E; ++r) b[r] = ld_global(psi + (size_t)(v + r * st.nb) * nx + m);
      } else {
#pragma unroll
        for (int r = 0; r < E; ++r) b[r] = x.at(m, v + r * st.nb);
        mix_twiddle<E, false>(b, wk);
        mix_dft<E, false>(b);
      }
      double s1 = 0.0, n1 = 0.0;
      if (td) {
        if (imag)
          col_kinetic<R, E, true, true, true>(b, v, st.nb, nx, jx, td, hp, hc, C{1, 0}, (const C*)nullptr, kspace, mid,
                                              want_s, s1, n1);
        else
          col_kinetic<R, E, true, false, true>(b, v, st.nb, nx, jx, td, hp, hc, C{1, 0}, (const C*)nullptr, kspace,
                                               mid, want_s, s1, n1);
      } else if (imag) {
        col_kinetic<R, E, false, true, true>(b, v, st.nb, nx, jx, nullptr, hp, hc, ld_global(kxt + jx), kyt, kspace,
                                             mid, want_s, s1, n1);
      } else {
        col_kinetic<R, E, false, false, true>(b, v, st.nb, nx, jx, nullptr, hp, hc, ld_global(kxt + jx), kyt, kspace,
                                              mid, want_s, s1, n1);
      }
      s_acc += s1;
      n_acc += n1;
      if (mid) {
        mix_dft<E, true>(b);
        mix_twiddle<E, true>(b, wk);
#pragma unroll
        for (int r = 0; r < E; ++r) x.at(m, v + r * st.nb) = b[r];
      } else {
#pragma unroll
        for (int r = 0; r < E; ++r) st_global(psi + (size_t)(v + r * st.nb) * nx + m, b[r]);
      }
    }
  });
  if (mid) {
    mix_inner_adj<true>(f, x);
    mix_first_adj<true, C>(f, x, [&](int m, int i, C a) { st_global(psi + (size_t)i * nx + m, a); });
  }
  double s[2] = {s_acc, n_acc};
  block_sum_thread0<2>(s, reinterpret_cast<double*>(twl + N));
  if (threadIdx.x == 0) {
    const int nt = nx / W;
    P.part[PART_S * 2 * nt + comp * nt + tile] = s[0];
    P.part[PART_NRM * 2 * nt + comp * nt + tile] = s[1];
  }
}

// -------------------------------------------------------------- row pass

// Offsets of a thread's points i0 + j step in an array of `end`; point 0 stands
// in for those past the end.
struct PointsAt {
  int i0, step, end;
  __device__ __forceinline__ size_t operator()(int j) const {
    const int i = i0 + j * step;
    return (size_t)(i < end ? i : i0);
  }
};

// `rows` rows (both components) of slot blockIdx.z, as row_pass_kernel.
// LDS: [rows][2][n] data, [n] twiddles. GENERAL as there.
template <typename R, bool GENERAL>
__global__ __launch_bounds__(kMixThreads) void mix_row_pass_kernel(const InstDev* __restrict__ insts,
                                                                   RunDev* __restrict__ runs, MixFft f,
                                                                   const typename Cx<R>::T* __restrict__ tw, int rows,
                                                                   unsigned div_n, int dur, int first_sub, int col_w) {
  typedef typename Cx<R>::T C;
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  RunDev& run = runs[inst];
  if (!run.active) return;
  const InstDev& P = insts[inst];
  const int N = f.n, ny = P.ny;
  const int y0 = blockIdx.x * rows;
  C* const psi = reinterpret_cast<C*>(P.psi) + (size_t)y0 * N;
  const size_t plane = (size_t)ny * N;
  MixTile<C> x;
  x.lds = reinterpret_cast<C*>(smem);
  C* const twl = x.lds + 2 * rows * N;
  x.tw = twl;
  x.batch = 2 * rows;  // transform m: row m / 2, component m % 2
  x.div_batch = 0;
  x.ms = N;
  x.is = 1;
  MixTwiddles<C> stw;
  stw.load(tw, N);
  mix_first<true, C>(f, x, [&](int m, int i) { return ld_global(psi + (m & 1) * plane + (size_t)(m >> 1) * N + i); });
  stw.store(tw, N, twl);
  const int nt2 = 2 * (N / col_w);
  if (blockIdx.x == 0) {
    if (first_sub) {
      const int step = run.step;
      record_pops(P, run.pops, run.pops_cap, step, nt2);
      if (threadIdx.x == 0) run.step = step + 1;
    }
    if (threadIdx.x == 0) run.form = FORM_HYBRID;
  }
  const double nrm = wave_sum_strided(P.part + PART_NRM * nt2, nt2);
  const double lam2 = P.atom_num / (P.dv_r * (double)N * (double)ny * nrm);
  mix_inner<true>(f, x);

  // Last stage in place, pointwise block over all points of the rows, two per
  // thread at a time (four: 233 registers, 10-35 % slower), adjoint last stage in place. With the block inside the
  // last stage (as the column pass has it) a thread held both components of up
  // to ten points: 256 registers, a third of the threads idle, and for dense
  // operators 30 KB of straight-line code per radix, whose fetching took longer
  // than its work on small grids. 96 x 100 complex128, dense: 20-28 -> 9 us;
  // 1000^2 dense 85-93 -> 46 us; 1000^2 fast path 44 -> 36 us (complex128) and 30
  // -> 22 us (complex64); 1536^2 complex128 is the exception (65 -> 92 us).
  const MixStage& st = f.st[f.ns - 1];
  const int items = st.nb * x.batch;
  mix_radix<kMixMidRadix>(st.radix, [&](auto rr) {
    constexpr int E = decltype(rr)::v;
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
      int m, v;
      x.item(st, w, &m, &v);
      C b[E];
#pragma unroll
      for (int r = 0; r < E; ++r) b[r] = x.at(m, v + r * st.nb);
      mix_twiddle<E, true>(b, x.tw + st.off + v * (E - 1));  // k = v: the span is n / radix
      mix_dft<E, true>(b);
#pragma unroll
      for (int r = 0; r < E; ++r) x.at(m, v + r * st.nb) = b[r];
    }
  });
  const double* vd0 = P.v_dense[0];
  const double* vd1 = P.v_dense[1];
  const C* px0 = vd0 ? nullptr : reinterpret_cast<const C*>(P.px[dur][0]);
  const C* px1 = vd1 ? nullptr : reinterpret_cast<const C*>(P.px[dur][1]);
  const C* qy0 = vd0 ? nullptr : reinterpret_cast<const C*>(P.py[dur][0]);
  const C* qy1 = vd1 ? nullptr : reinterpret_cast<const C*>(P.py[dur][1]);
  const C* eth = reinterpret_cast<const C*>(P.etheta);
  const RowCoef<R> k(P, dur, lam2);
  const int points = rows * N;
  __syncthreads();
  for (int i0 = threadIdx.x; i0 < points; i0 += 2 * (int)blockDim.x) {
    const PointsAt offset{i0, (int)blockDim.x, points};
    C a0[2], a1[2], tx0[2], tx1[2], tex[2], py0[2], py1[2];
    int at[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = (int)offset(j);
      const int row = mix_div(i, N, div_n), xx = i - row * N;
      at[j] = i + row * N;  // (2 row) n + xx
      tx0[j] = px0 ? ld_global(px0 + xx) : C{1, 0};
      tx1[j] = px1 ? ld_global(px1 + xx) : C{1, 0};
      tex[j] = ld_global(eth + xx);
      py0[j] = qy0 ? ld_global(qy0 + y0 + row) : C{1, 0};
      py1[j] = qy1 ? ld_global(qy1 + y0 + row) : C{1, 0};
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a0[j] = x.lds[at[j]];
      a1[j] = x.lds[at[j] + N];
    }
    row_pointwise<R, 2, !GENERAL>(a0, a1, P, k, (size_t)y0 * N, offset, py0, py1, tx0, tx1, tex);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      x.lds[at[j]] = a0[j];
      x.lds[at[j] + N] = a1[j];
    }
  }
  __syncthreads();
  mix_radix<kMixMidRadix>(st.radix, [&](auto rr) {
    constexpr int E = decltype(rr)::v;
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
      int m, v;
      x.item(st, w, &m, &v);
      C b[E];
#pragma unroll
      for (int r = 0; r < E; ++r) b[r] = x.at(m, v + r * st.nb);
      mix_dft<E, false>(b);
      mix_twiddle<E, false>(b, x.tw + st.off + v * (E - 1));
#pragma unroll
      for (int r = 0; r < E; ++r) x.at(m, v + r * st.nb) = b[r];
    }
  });
  mix_inner_adj<false>(f, x);
  mix_first_adj<false, C>(f, x, [&](int m, int i, C a) {
    st_global(psi + (m & 1) * plane + (size_t)(m >> 1) * N + i, a);
  });
}

// ---------------------------------------------------- standalone fft_2d
// The transform of `batch` rows (ROWS) or columns of array blockIdx.z of the
// pair (in place allowed); rows take the factor (-1)^(x+y) * scale before
// (forward) or after (inverse), as fft_rows_kernel.
template <typename R, bool ROWS, bool INV>
__global__ __launch_bounds__(kMixThreads) void mix_fft_kernel(FftPair io, MixFft f,
                                                              const typename Cx<R>::T* __restrict__ tw, int nx,
                                                              int batch, unsigned div_batch, double scale) {
  typedef typename Cx<R>::T C;
  extern __shared__ double smem[];
  const int N = f.n;
  const int t0 = (ROWS ? (int)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x)) * batch;
  const size_t base = ROWS ? (size_t)t0 * N : (size_t)t0;
  const C* in = reinterpret_cast<const C*>(io.in[blockIdx.z]) + base;
  C* out = reinterpret_cast<C*>(io.out[blockIdx.z]) + base;
  const size_t es = ROWS ? 1 : nx, ms = ROWS ? N : 1;  // strides of element and transform in global memory
  MixTile<C> x;
  x.lds = reinterpret_cast<C*>(smem);
  C* const twl = x.lds + batch * N;
  x.tw = twl;
  x.batch = batch;
  x.div_batch = div_batch;
  x.ms = ROWS ? N : 1;
  x.is = ROWS ? 1 : batch;
  const R sc = (R)scale;
  auto factor = [&](int m, int i) -> R { return ((t0 + m + i) & 1) ? -sc : sc; };
  MixTwiddles<C> stw;
  stw.load(tw, N);
  mix_first<INV, C>(f, x, [&](int m, int i) {
    const C a = ld_global(in + m * ms + i * es);
    return ROWS && !INV ? cscale(a, factor(m, i)) : a;
  });
  stw.store(tw, N, twl);
  mix_inner<INV>(f, x);
  const MixStage& st = f.st[f.ns - 1];
  const int items = st.nb * batch;
  mix_radix<kMixMidRadix>(st.radix, [&](auto rr) {
    constexpr int E = decltype(rr)::v;
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
      int m, v;
      x.item(st, w, &m, &v);
      C b[E];
#pragma unroll
      for (int r = 0; r < E; ++r) b[r] = x.at(m, v + r * st.nb);
      mix_twiddle<E, INV>(b, x.tw + st.off + v * (E - 1));
      mix_dft<E, INV>(b);
#pragma unroll
      for (int r = 0; r < E; ++r) {
        const int i = v + r * st.nb;
        st_global(out + m * ms + i * es, ROWS && INV ? cscale(b[r], factor(m, i)) : b[r]);
      }
    }
  });
}

enum { MIX_COL, MIX_ROW, MIX_ROW_GENERAL, MIX_FFT_COLS, MIX_FFT_COLS_INV, MIX_FFT_ROWS, MIX_FFT_ROWS_INV };

// Launchers and kernel addresses, instantiated per precision
// (sgpe_mixed_f64.hip, sgpe_mixed_f32.hip).
template <typename R> struct MixKernels {
  static void col(dim3 g, dim3 b, size_t l, hipStream_t s, hipEvent_t e0, hipEvent_t e1, const InstDev* i, RunDev* r,
                  const MixFft& f, const void* tw, int w, unsigned div_w, int mode, int dp, int dc);
  static void row(dim3 g, dim3 b, size_t l, hipStream_t s, hipEvent_t e0, hipEvent_t e1, const InstDev* i, RunDev* r,
                  const MixFft& f, const void* tw, int rows, unsigned div_n, int dur, int first, int col_w, bool general);
  static void fft(dim3 g, dim3 b, size_t l, hipStream_t s, FftPair io, const MixFft& f, const void* tw, int nx,
                  int batch, unsigned div_batch, bool rows, bool inv, double scale);
  static const void* kernel(int which);
};

}  // namespace sgpe
