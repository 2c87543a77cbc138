// Split-step kernels. One split step (the reference's full_step,
// spinor_gpe/pspinor/tensor_propagator.py:214-222) is three sub-steps; each
// sub-step here is two sweeps over the state:
//
//   column pass  (per column jx, per component; y is the strided axis)
//       DFT_y -> K_prev (end of the previous sub-step) -> [S: sum |.|^2]
//             -> K_cur (start of this sub-step) -> [NRM: sum |.|^2] -> IDFT_y
//   row pass     (per row y, both components together)
//       IDFT_x -> normalize (from NRM) -> U C P C U -> DFT_x * dx dy/(2 pi)
//
// which is tensor_propagator.py:242-271 with the fftshift/ifftshift pairs and
// the FFT scale factors folded away: for even grid sizes the shifts only
// multiply real space by (-1)^(x+y), which commutes with every real-space
// factor, and the scale is absorbed by the renormalization that follows each
// inverse transform. The k-space renormalization at the end of a sub-step
// (tensor_propagator.py:271) is deferred: the next real-space renormalization
// absorbs it, the per-step populations are ratios of the S sums, and the
// explicit normalize kernel applies it when the state is handed back.
#pragma once

#include "sgpe_fft.h"

namespace sgpe {

// ---------------------------------------------------------------- helpers

// sin and cos by Cody-Waite reduction x = k pi/2 + r, |r| <= pi/4, with
// pi/2 = P1 + P2 + P3 (P1 pi/2 rounded to double, P2 and P3 the successive
// remainders): each fma(-k, Pi, r) rounds once, so r is within a few 1e-16
// of x - k pi/2 for |k| < 1e15 (|x| < 1.5e15; beyond, a double no longer
// resolves a radian of phase and the error grows with |x|). The quadrant is
// k mod 4, computed exactly in double. Then polynomials in r (sc_poly:
// truncation below half an ulp); within 2 ulp of the correctly rounded values. There is no
// library fallback: inlined at every call site, the device library's
// large-argument code made the row pass's pointwise block twice as slow even
// where it never ran (instruction fetch across it).
__device__ __forceinline__ double cw_reduce(double x, int* quadrant) {
  const double k = rint(x * 0.6366197723675814);
  double r = fma(-k, 1.5707963267948966, x);
  r = fma(-k, 6.123233995736766e-17, r);
  r = fma(-k, -1.4973849048591698e-33, r);
  *quadrant = (int)fma(-4.0, floor(k * 0.25), k);
  return r;
}

template <typename R> __device__ __forceinline__ void quadrant_fix(int q, R sr, R cr, R* s, R* c) {
  const R ss = (q & 1) ? cr : sr;
  const R cc = (q & 1) ? sr : cr;
  *s = (q & 2) ? -ss : ss;
  *c = ((q + 1) & 2) ? -cc : cc;
}

// sin and cos for |r| <= pi/4. Double: minimax polynomials (Remez exchange,
// relative error with the rounded coefficients 5.9e-18 of sin, 1.2e-18 of cos;
// 2^-53-rounding dominates: largest error 7.4e-17 and 9.6e-17, as the Taylor series with four
// more terms has). Float: Taylor terms through r^9 / r^10.
__device__ __forceinline__ void sc_poly(double r, double* s, double* c) {
  const double r2 = r * r;
  double ps = 1.5896827972044486e-10;
  ps = fma(ps, r2, -2.5050758654058057e-08);
  ps = fma(ps, r2, 2.7557313695231825e-06);
  ps = fma(ps, r2, -0.00019841269829816967);
  ps = fma(ps, r2, 0.008333333333322425);
  ps = fma(ps, r2, -0.16666666666666632);
  *s = fma(r * r2, ps, r);
  double pc = -1.1359669918955859e-11;
  pc = fma(pc, r2, 2.0875723685357163e-09);
  pc = fma(pc, r2, -2.7557314355247977e-07);
  pc = fma(pc, r2, 2.4801587289491845e-05);
  pc = fma(pc, r2, -0.0013888888888874139);
  pc = fma(pc, r2, 0.0416666666666666);
  pc = fma(pc, r2, -0.5);
  *c = fma(r2, pc, 1.0);
}
__device__ __forceinline__ void sc_poly(float r, float* s, float* c) {
  const float r2 = r * r;
  float ps = 2.7557319223985893e-06f;
  ps = fmaf(ps, r2, -0.0001984126984126984f);
  ps = fmaf(ps, r2, 0.008333333333333333f);
  ps = fmaf(ps, r2, -0.16666666666666666f);
  *s = fmaf(r * r2, ps, r);
  float pc = -2.755731922398589e-07f;
  pc = fmaf(pc, r2, 2.48015873015873e-05f);
  pc = fmaf(pc, r2, -0.001388888888888889f);
  pc = fmaf(pc, r2, 0.041666666666666664f);
  pc = fmaf(pc, r2, -0.5f);
  *c = fmaf(r2, pc, 1.0f);
}

// The reduction runs in double for every argument, also in complex64 (exact
// for any float x): a single-precision reduction for small arguments with the
// double one as a fallback put two branches around every sin/cos, and the
// blocks they cut the pointwise code into kept its independent sin/cos chains
// from overlapping (the complex64 real-time row pass took 0.3 us longer).
template <typename R> __device__ __forceinline__ void sc(R x, R* s, R* c) {
  int q;
  R sr, cr;
  sc_poly((R)cw_reduce((double)x, &q), &sr, &cr);
  quadrant_fix<R>(q, sr, cr, s, c);
}
template <typename R> __device__ __forceinline__ R ex(R x);
template <> __device__ __forceinline__ double ex<double>(double x) { return exp(x); }
template <> __device__ __forceinline__ float ex<float>(float x) { return expf(x); }

// exp(x) for |x| <= kSmallExp: minimax polynomial of (exp(x) - 1 - x) / x^2
// (Remez exchange; relative error with the rounded coefficients 1.4e-17 double,
// 5.2e-9 float, largest error after rounding 1.2e-16 and 6.2e-8). No reduction
// and no scaling.
__device__ __forceinline__ double ex_poly(double x) {
  double p = 2.5117848056977748e-08;
  p = fma(p, x, 2.7631276855506471e-07);
  p = fma(p, x, 2.7557216339313716e-06);
  p = fma(p, x, 2.4801489951255983e-05);
  p = fma(p, x, 0.0001984126991734402);
  p = fma(p, x, 0.0013888888947006998);
  p = fma(p, x, 0.008333333333307221);
  p = fma(p, x, 0.04166666666651544);
  p = fma(p, x, 0.166666666666667);
  p = fma(p, x, 0.5000000000000013);
  return fma(x, fma(p, x, 1.0), 1.0);
}
__device__ __forceinline__ float ex_poly(float x) {
  float p = 0.0013950489013913796f;
  p = fmaf(p, x, 0.0083688876559632787f);
  p = fmaf(p, x, 0.04166620583338496f);
  p = fmaf(p, x, 0.16666518853794891f);
  p = fmaf(p, x, 0.5000000095175364f);
  return fmaf(x, fmaf(p, x, 1.0f), 1.0f);
}

// Arguments up to these bounds take the polynomials without a reduction
// (SMALL below): the reduced argument is then x itself and the quadrant 0, so
// sin and cos come out bit-identical either way.
constexpr double kSmallAngle = 0.785;
constexpr double kSmallExp = 0.346;

// exp(-i E Delta) for Delta = dt (real time) or -i dt (imaginary time).
template <typename R, bool IMAG, bool SMALL = false>
__device__ __forceinline__ typename Cx<R>::T phase_op(R e_dt) {
  typedef typename Cx<R>::T C;
  if constexpr (IMAG) {
    return C{SMALL ? ex_poly(-e_dt) : ex<R>(-e_dt), (R)0};
  } else {
    R s, c;
    if constexpr (SMALL)
      sc_poly(-e_dt, &s, &c);
    else
      sc<R>(-e_dt, &s, &c);
    return C{c, s};
  }
}

// p times a phase factor from phase_op: in imaginary time the factor is
// real (zero imaginary part), and scaling by its real part gives the same
// result as the complex product without its multiplications by zero.
template <bool IMAG, typename C> __device__ __forceinline__ C mul_phase(C p, C u) {
  if constexpr (IMAG)
    return cscale(p, u.x);
  else
    return cmul(p, u);
}

// The pass kernels select their pointwise code by uniform flags (time mode,
// dense or separable operators) OUTSIDE the loops, in separately compiled
// variants: inside one loop the compiler would evaluate the sin/cos or exp
// of every alternative for every point and select afterwards.

// The same with a non-temporal hint, for the streaming flags of
// sgpe_plan_set_streaming. The compiler merges the two arms of the passes'
// run-time choice into one without the hint, so that the flags have no effect at
// present (kept apart by force: 3 % of a 512^2 complex128 step gained, batched
// 1024^2 complex64 70 % slower).
template <typename C> __device__ __forceinline__ C ld_stream(const C* p) {
  typedef decltype(p->x) S;
  typedef S V2 __attribute__((ext_vector_type(2)));
  const V2 w = __builtin_nontemporal_load((const __attribute__((address_space(1))) V2*)p);
  return C{w.x, w.y};
}
template <typename C> __device__ __forceinline__ void st_stream(C* p, C v) {
  typedef decltype(v.x) S;
  typedef S V2 __attribute__((ext_vector_type(2)));
  const V2 w = {v.x, v.y};
  __builtin_nontemporal_store(w, (__attribute__((address_space(1))) V2*)p);
}

// Device-coherent accesses (cache policy SC1: device scope) to data that
// other workgroups of the same launch write or read, through a buffer
// resource over [base, base + bytes): writes reach the device's coherence
// point before the wave's vmcnt drains, and reads do not return lines an
// L2 of another XCD may hold stale, so workgroups of one launch exchange
// data without cache-wide writebacks or invalidations. Out-of-range offsets
// read 0 and drop writes (the resource's bound). 0x00020000 is the
// resource's third word for gfx9 targets (raw buffer, 32-bit data format).
constexpr int kCpolSc1 = 16;
struct CoherentBuf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ CoherentBuf(void* base, uint32_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(base, 0, (int)bytes, 0x00020000)) {}
  template <typename C> __device__ __forceinline__ C load(uint32_t off) const {
    if constexpr (sizeof(C) == 16) {
      typedef unsigned int V4 __attribute__((ext_vector_type(4)));
      const V4 w = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, kCpolSc1);
      return __builtin_bit_cast(C, w);
    } else {
      typedef unsigned int V2 __attribute__((ext_vector_type(2)));
      const V2 w = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, kCpolSc1);
      return __builtin_bit_cast(C, w);
    }
  }
  template <typename C> __device__ __forceinline__ void store(uint32_t off, C v) const {
    if constexpr (sizeof(C) == 16) {
      typedef unsigned int V4 __attribute__((ext_vector_type(4)));
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(V4, v), r, (int)off, 0, kCpolSc1);
    } else {
      typedef unsigned int V2 __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, v), r, (int)off, 0, kCpolSc1);
    }
  }
};
// Access modes of the pass bodies (CM): device-coherent state and partial
// sum reads (CM_LOAD) and writes (CM_STORE); 0 = ordinary accesses.
enum { CM_LOAD = 1, CM_STORE = 2 };
__device__ __forceinline__ double ld_coherent(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coherent(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sum of n doubles by one wave: lane l adds entries l, l + 64, ..., then a
// butterfly across the lanes; every lane gets the same total, and every wave
// that calls it sums in the same order. COH: device-coherent reads.
// Entries are read four per lane at a time, so that their loads are in flight
// together (one load per iteration made every entry a dependent memory round
// trip), and added in the same order as one at a time.
template <bool COH = false>
__device__ __forceinline__ double wave_sum_strided(const double* __restrict__ p, int n) {
  const int lane = threadIdx.x & 63;
  double v = 0.0;
  for (int i = lane; i < n; i += 4 * 64) {
    double e[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int ik = i + 64 * k;
      e[k] = ik < n ? (COH ? ld_coherent(p + ik) : ld_global(p + ik)) : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (i + 64 * k < n) v += e[k];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The same sum with the loads of the first 256 entries issued by the
// constructor and the rest done by sum(): a row pass issues them ahead of its
// state loads. Loads return in order, so the norm, its reduction across the
// lanes, the division and the square root then finish while the state is still
// on its way; loaded after the state, all of it came on top. Same order of
// additions, same result.
struct PartSum {
  const double* __restrict__ p;
  int n;
  double e[4];
  __device__ __forceinline__ PartSum(const double* __restrict__ part, int count) : p(part), n(count) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < 4; ++k) e[k] = ld_global(p + (lane + 64 * k < n ? lane + 64 * k : 0));
  }
  __device__ __forceinline__ double sum() const {
    const int lane = threadIdx.x & 63;
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (lane + 64 * k < n) v += e[k];
    for (int i = lane + 256; i < n; i += 4 * 64) {
      double f[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] = i + 64 * k < n ? ld_global(p + i + 64 * k) : 0.0;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (i + 64 * k < n) v += f[k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
  }
};

template <typename R> __device__ __forceinline__ double norm2d(typename Cx<R>::T a) {
  double x = (double)a.x, y = (double)a.y;
  return x * x + y * y;
}

// ------------------------------------------------------------ column pass

// Workgroups are dealt to the 8 XCDs (each with its own L2) round-robin in
// dispatch order. With n tiles a multiple of 8, XCD k gets the contiguous
// tiles [k n/8, (k+1) n/8), so neighbouring column tiles, which share cache
// lines when a tile row is narrower than a line (complex64, 8 columns),
// meet in one L2 instead of being fetched twice.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_tile(int b, int n) {
  return n % kXcds == 0 ? (b % kXcds) * (n / kXcds) + b / kXcds : b;
}

// Kinetic factors of the column pass on this thread's E points t + j T of column jx:
// the closing K of the previous sub-step (unless the state is already in
// k-space: `kspace`) and the opening K of this one (`mid`), with the norm sums.
// S is the norm between the two, NRM the one after both; want_s: S is asked
// for (populations, once a full step).
//  - Real time: |K| = 1, so S = NRM, and both half steps are one phase from one
//    pair of tables (k2x, k2y): 10 instructions a point where the two factors
//    and two sums took 22.
//  - Imaginary time: both K are real; the tables hold them as the parts of one
//    entry, and without S their product is applied at once (8 instructions).
// DENSE: K from the dense T array. kx, ky: the table values of this column and
// the y table (KYG: in global memory, else staged in LDS); in real time with
// the state in k-space they are those of K_cur alone.
// The uniform choices are taken around whole point loops: tested per point,
// they put every table read in a block of its own with its own wait, a chain
// of dependent LDS round trips.
template <typename R, int E, bool DENSE, bool IMAG, bool KYG, typename C>
__device__ __forceinline__ void col_kinetic(C (&a)[E], int t, int T, int nx, int jx, const double* __restrict__ td, R hp,
                                            R hc, C kx, const C* ky, bool kspace, bool mid, bool want_s,
                                            double& s_acc, double& n_acc) {
  auto yval = [&](int j) -> C { return KYG ? ld_global(ky + t + j * T) : ky[t + j * T]; };
  auto dense = [&](int j, R h) -> C {
    return phase_op<R, IMAG>((R)ld_global(td + (size_t)(t + j * T) * nx + jx) * h);
  };
  if (kspace && !mid) {
#pragma unroll
    for (int j = 0; j < E; ++j) n_acc += norm2d<R>(a[j]);
    s_acc = n_acc;
    return;
  }
  if constexpr (!IMAG) {
    const R h = (kspace ? (R)0 : hp) + (mid ? hc : (R)0);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      C k;
      if constexpr (DENSE)
        k = dense(j, h);
      else
        k = cmul(kx, yval(j));
      a[j] = cmul(a[j], k);
      n_acc += norm2d<R>(a[j]);
    }
    s_acc = n_acc;
  } else if (mid && want_s && !kspace) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      R k1, k2;
      if constexpr (DENSE) {
        k1 = dense(j, hp).x;
        k2 = dense(j, hc).x;
      } else {
        const C y = yval(j);
        k1 = kx.x * y.x;
        k2 = kx.y * y.y;
      }
      a[j] = cscale(a[j], k1);
      s_acc += norm2d<R>(a[j]);
      a[j] = cscale(a[j], k2);
      n_acc += norm2d<R>(a[j]);
    }
  } else {
    if (kspace) {
#pragma unroll
      for (int j = 0; j < E; ++j) s_acc += norm2d<R>(a[j]);
    }
    const R h = (kspace ? (R)0 : hp) + (mid ? hc : (R)0);
    // One factor a point: K_prev K_cur, or one of them with 1 for the other.
    const R x1 = kspace ? (R)1 : kx.x, x2 = mid ? kx.y : (R)1;
    const R x12 = x1 * x2;
#pragma unroll
    for (int j = 0; j < E; ++j) {
      R k;
      if constexpr (DENSE) {
        k = dense(j, h).x;
      } else {
        const C y = yval(j);
        k = x12 * ((kspace ? (R)1 : y.x) * (mid ? y.y : (R)1));
      }
      a[j] = cscale(a[j], k);
      n_acc += norm2d<R>(a[j]);
    }
    if (!kspace) s_acc = n_acc;
  }
}

// One column tile of one component (the body of col_pass_kernel and of the
// persistent step kernel). `gate` is called once every global load of the
// prologue has been issued: it returns -1 to drop the tile (inactive slot),
// else whether the stored state is already in k-space (1) or hybrid (0).
// DENSE: the plan has some slot with a dense kinetic array (the code then
// also handles table slots); otherwise every slot uses the separable tables.
template <typename R, int N, int E, int W, bool DENSE, int CM, class Gate, bool GKY = false>
__device__ __forceinline__ void col_item(const InstDev& P, typename Cx<R>::T* __restrict__ psi, int nx,
                                         const typename Cx<R>::T* __restrict__ tws, int mode, int d_prev,
                                         int d_cur, int stream, int comp, int tile, double* smem, Gate gate) {
  typedef typename Cx<R>::T C;
  typedef LdsView<W, 1 << 30, 0> V;
  constexpr int T = N / E;
  // LDS: [W*N exchange][N twiddles][N y phase table][sums] (tables and a
  // separate sum slot when they fit). GKY: the y phase table stays in global
  // memory (cache resident) even where it would fit, which leaves LDS for more
  // workgroups per CU in batched plans.
  constexpr size_t kData = (size_t)W * N * sizeof(C);
  constexpr bool kTw = tw_in_lds(kData, N, sizeof(C));
  constexpr bool kKy = !GKY && kTw && kData + 2 * (size_t)N * sizeof(C) <= kLdsBytes;
  constexpr size_t kBase = kData + (kTw ? (size_t)N * sizeof(C) : 0) + (kKy ? (size_t)N * sizeof(C) : 0);
  constexpr bool kSumSep = col_sum_separate(kBase);
  // The W*T threads of a tile interleave its W columns, so a column's
  // transform lies within one wave when the whole tile does.
  constexpr bool kWave = W * T <= 64;
  const int c = threadIdx.x % W;
  const int t = threadIdx.x / W;
  const int jx = tile * W + c;
  C* const sm = reinterpret_cast<C*>(smem);
  C* lds = sm + c;
  C* col = psi + (size_t)comp * N * nx + jx;

  // Every global load is issued before any computation: the state first,
  // then the kinetic tables and twiddles (staged into LDS).
  constexpr int kBlock = W * T;
  C a[E];
  // CM & CM_LOAD / CM_STORE: device-coherent state reads / writes; element
  // (comp, jy, jx) at byte ((comp N + jy) nx + jx) sizeof(C)
  const CoherentBuf cb(psi, CM ? (uint32_t)(2 * (size_t)N * nx * sizeof(C)) : 0u);
  const uint32_t cbase = (uint32_t)(((size_t)comp * N * nx + jx) * sizeof(C));
  if constexpr ((CM & CM_LOAD) != 0) {
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = cb.load<C>(cbase + (uint32_t)((t + j * T) * nx * sizeof(C)));
  } else if (stream) {
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = ld_stream(col + (size_t)(t + j * T) * nx);
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = ld_global(col + (size_t)(t + j * T) * nx);
  }
  const double* td = P.t_dense[comp];
  const bool mid = mode != COL_EXIT;
  const bool imag = P.imag != 0;
  C kx = C{(R)1, (R)0};
  TableStage<kKy, N, kBlock, C> sky;
  TableStage<kTw, N, kBlock, C> stw;
  // Both half steps' tables; the closing pass in real time takes K_prev's.
  const bool one = !mid && !imag;
  if (!td) kx = ld_global(reinterpret_cast<const C*>(one ? P.kx[d_prev][comp] : P.k2x[d_prev][d_cur][comp]) + jx);
  // The y table is staged unconditionally (a conditional fill puts the
  // staging registers in scratch); without it (dense kinetic operator) the
  // twiddle table, also N entries, stands in and the copy goes unused.
  sky.load(td ? tws : reinterpret_cast<const C*>(one ? P.ky[d_prev][comp] : P.k2y[d_prev][d_cur][comp]));
  stw.load(tws);
  const int gk = gate();
  if (gk < 0) return;
  const bool kspace = gk != 0;
  const C* ky = sky.store(sm + W * N + N);
  const C* tw = stw.store(sm + W * N);

  if (!kspace) {
    if constexpr (kWave && (kTw || kKy)) __syncthreads();  // publishes the staged tables
    if constexpr (kTw) {
      fft_run<N, E, false, V, kWave>(a, t, tw, lds);
    } else {
      const StageTwiddles<N, E, 1, C> none{};
      fft_run_pre<N, E, false, V, kWave>(a, t, tw, lds, none);
    }
  } else {
    __syncthreads();  // publishes the staged tables
  }

  double s_acc = 0.0, n_acc = 0.0;
  const R hp = (R)(0.5 * P.dt_sub[d_prev]);
  const R hc = (R)(0.5 * P.dt_sub[d_cur]);
  const bool want_s = mode == COL_MID_S;
  if (!DENSE || !td) {
    if (imag) {
      col_kinetic<R, E, false, true, !kKy>(a, t, T, nx, jx, nullptr, hp, hc, kx, ky, kspace, mid, want_s, s_acc, n_acc);
    } else if (kspace) {  // first pass from k-space: K_cur's own tables
      const C kc = ld_global(reinterpret_cast<const C*>(P.kx[d_cur][comp]) + jx);
      col_kinetic<R, E, false, false, true>(a, t, T, nx, jx, nullptr, hp, hc, kc,
                                               reinterpret_cast<const C*>(P.ky[d_cur][comp]), true, mid, want_s,
                                               s_acc, n_acc);
    } else {
      col_kinetic<R, E, false, false, !kKy>(a, t, T, nx, jx, nullptr, hp, hc, kx, ky, false, mid, want_s, s_acc,
                                               n_acc);
    }
  } else if constexpr (DENSE) {
    if (imag)
      col_kinetic<R, E, true, true, !kKy>(a, t, T, nx, jx, td, hp, hc, kx, ky, kspace, mid, want_s, s_acc, n_acc);
    else
      col_kinetic<R, E, true, false, !kKy>(a, t, T, nx, jx, td, hp, hc, kx, ky, kspace, mid, want_s, s_acc, n_acc);
  }
  // Columns of 1024 points and more, and complex64 columns: an opaque copy of
  // t for the inverse transform and the stores, so their addresses are
  // recomputed rather than held since the loads (as in row_item; 2-5 % per
  // pass at 1024 points and more; complex64 512-point columns 82 -> 60
  // registers, 8 waves per SIMD instead of 5).
  int tf = t;
  if constexpr (N >= 1024 || sizeof(C) == 8) asm volatile("" : "+v"(tf));
  if (mid) {
    if constexpr (kTw) {
      fft_run<N, E, true, V, kWave>(a, tf, tw, lds);
    } else {
      const StageTwiddles<N, E, 1, C> none{};
      fft_run_pre<N, E, true, V, kWave>(a, tf, tw, lds, none);
    }
  }
  if constexpr ((CM & CM_STORE) != 0) {
#pragma unroll
    for (int j = 0; j < E; ++j) cb.store<C>(cbase + (uint32_t)((tf + j * T) * nx * sizeof(C)), a[j]);
  } else if (stream) {
#pragma unroll
    for (int j = 0; j < E; ++j) st_stream(col + (size_t)(tf + j * T) * nx, a[j]);
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) st_global(col + (size_t)(tf + j * T) * nx, a[j]);
  }

  // S differs from NRM only in imaginary time with both factors present; one
  // sum otherwise.
  double v[2] = {s_acc, n_acc};
  double* const sums = kSumSep ? reinterpret_cast<double*>(reinterpret_cast<char*>(smem) + kBase) : smem;
  if (imag && mid && (want_s || kspace)) {
    if constexpr (kSumSep)
      block_sum_thread0<2>(v, sums);
    else
      block_sum<2>(v, sums);
  } else {
    double w[1] = {n_acc};
    if constexpr (kSumSep)
      block_sum_thread0<1>(w, sums);
    else
      block_sum<1>(w, sums);
    v[0] = v[1] = w[0];
  }
  if (threadIdx.x == 0) {
    const int nt = nx / W;
    double* ps = P.part + PART_S * 2 * nt + comp * nt + tile;
    double* pn = P.part + PART_NRM * 2 * nt + comp * nt + tile;
    if constexpr ((CM & CM_STORE) != 0) {
      st_coherent(ps, v[0]);
      st_coherent(pn, v[1]);
    } else {
      *ps = v[0];
      *pn = v[1];
    }
  }
}

template <typename R, int N, int E, int W, bool DENSE, bool GKY = false>
__global__ __launch_bounds__(W*(N / E)) void col_pass_kernel(const InstDev* __restrict__ insts,
                                                             RunDev* __restrict__ runs, void* direct_psi,
                                                             int direct_n, const typename Cx<R>::T* __restrict__ tws,
                                                             int mode, int d_prev, int d_cur, int stream) {
  typedef typename Cx<R>::T C;
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  const InstDev& P = insts[inst];
  // A single-slot plan passes its state's address and row length as kernel
  // arguments (direct_psi): the state loads are issued at once and the
  // active flag is checked after them. Otherwise the address and length are
  // read together with the active flag, so the state loads wait for one
  // round of scalar loads, not two.
  const bool direct = direct_psi != nullptr;
  C* const psi = reinterpret_cast<C*>(direct ? direct_psi : P.psi);
  const int nx = direct ? direct_n : P.nx;
  if (!direct && (!runs[inst].active || !psi || nx <= 0)) return;
  auto gate = [&]() -> int {
    if (direct) {
      // The prologue loads stay ahead of the flag test (an inactive slot's
      // state and tables are still allocated: the host passes direct_psi
      // only for a loaded slot).
      asm volatile("" ::: "memory");
      if (!runs[inst].active) return -1;
    }
    return runs[inst].form == FORM_KSPACE ? 1 : 0;
  };
  col_item<R, N, E, W, DENSE, 0, decltype(gate), GKY>(P, psi, nx, tws, mode, d_prev, d_cur, stream, blockIdx.y,
                                     xcd_tile(blockIdx.x, nx / W), smem, gate);
}

// Sum of one partial slot over all column tiles of both components
// (deterministic: same order in every block). All threads get the result.
__device__ __forceinline__ void part_sums(const double* part, int nt2, int slot, int split, double* out2,
                                          double* scratch) {
  double v[2] = {0.0, 0.0};
  const double* p = part + (size_t)slot * nt2;
  for (int i = threadIdx.x; i < nt2; i += blockDim.x) v[(split && i >= nt2 / 2) ? 1 : 0] += p[i];
  block_sum<2>(v, scratch);
  out2[0] = v[0];
  out2[1] = v[1];
}

// Real-space block of the row pass, U C P C U with the normalization folded in
// (tensor_propagator.py:244-267), on this thread's points J0 <= j < J1 of row
// y, both components. The row passes of batched complex64 plans are bound by
// the number of vector instructions they issue (four cycles each for a wave,
// in float as in double), the transforms' about half of them, so this block is
// written for few:
//  - Every slot-uniform factor is formed once per row (RowCoef): the interaction
//    phases take the unnormalized densities, and the normalization and the
//    forward transform's scale ride in the first coupling factor.
//  - C = [[a, b e^{-i theta}], [b e^{i theta}, a]] has b imaginary in real time
//    and real in imaginary time: b e^{-i theta} takes two multiplications, C
//    three fused operations per output part. (Applying e^{-i theta} to psi_1
//    on both sides of a theta-free C takes two operations less, but there the
//    table's rounded modulus multiplies all of psi_1 in every sub-step instead
//    of the coupled part alone: over 20000 complex64 steps the fidelity with
//    complex128 fell from 0.97 to 0.93.)
//  - In imaginary time U and P are real factors.
//  - Where the phases of all points of a wave are small (they are g n dt / 2:
//    about 1e-2), their sin/cos or exp is a polynomial alone; one wave-uniform
//    test chooses the code for the whole block (SMALL). Tested per point, it
//    would cut the block into pieces that cannot overlap. Phases of dense
//    potentials and couplings are judged once, on the host (dense_small).
// Row pass before and after (dispatch times, us): 8 x 1024^2 complex64
// imaginary time 75.5 -> 69.6, 16 x 512^2 complex64 imaginary 38.2 -> 35.6, one
// 2048^2 complex128 real 86.9 -> 83.1, one 512^2 real 10.7 -> 10.2 (complex128)
// and 7.9 -> 7.3 (complex64).
template <typename R> struct RowCoef {
  bool imag, theta, dense_small;
  R kuu, kdd, kud;  // interaction phase of U per unnormalized density
  R sc;             // normalization x forward transform scale
  R ca, cb;         // a and b of C (b: its imaginary part in real time)
  R dts;            // sub-step
  __device__ __forceinline__ RowCoef(const InstDev& P, int dur, double lam2) {
    const double h = 0.5 * P.dt_sub[dur] * lam2;
    imag = P.imag != 0;
    theta = P.theta_x != nullptr;
    dense_small = P.dense_small != 0;
    kuu = (R)(P.g_uu * h);
    kdd = (R)(P.g_dd * h);
    kud = (R)(P.g_ud * h);
    sc = (R)(sqrt(lam2) * P.fft_c);
    ca = (R)P.c_alpha[dur];
    cb = (R)(imag ? P.c_beta_re[dur] : P.c_beta_im[dur]);
    dts = (R)P.dt_sub[dur];
  }
};

// (p0, p1) <- [[a, b e], [b conj(e), a]] (p0, p1) with b times i in real time;
// s = b Re(e), r = b Im(e). NT: e = 1 (r unused). a is close to 1: its product
// is the one that is not rounded by itself (rounded, p (1 - 1e-7) loses the
// same part of an ulp at every point of the same mantissa, and the populations
// of a complex64 run drifted by 2e-8 a sub-step).
template <bool IMAG, bool NT, typename C, typename R>
__device__ __forceinline__ void mix(C& p0, C& p1, R a, R s, R r) {
  C q0, q1;
  if constexpr (NT) {
    static_assert(IMAG, "theta-free form: imaginary time");
    q0 = C{fma(a, p0.x, s * p1.x), fma(a, p0.y, s * p1.y)};
    q1 = C{fma(a, p1.x, s * p0.x), fma(a, p1.y, s * p0.y)};
  } else if constexpr (IMAG) {
    q0 = C{fma(a, p0.x, fma(s, p1.x, -r * p1.y)), fma(a, p0.y, fma(s, p1.y, r * p1.x))};
    q1 = C{fma(a, p1.x, fma(s, p0.x, r * p0.y)), fma(a, p1.y, fma(s, p0.y, -r * p0.x))};
  } else {
    q0 = C{fma(a, p0.x, -fma(s, p1.y, r * p1.x)), fma(a, p0.y, fma(s, p1.x, -r * p1.y))};
    q1 = C{fma(a, p1.x, fma(-s, p0.y, r * p0.x)), fma(a, p1.y, fma(s, p0.x, r * p0.y))};
  }
  p0 = q0;
  p1 = q1;
}

// Interaction phases of one point.
template <typename R, typename C>
__device__ __forceinline__ void point_phases(C p0, C p1, const RowCoef<R>& k, R* e0, R* e1) {
  const R m0 = p0.x * p0.x + p0.y * p0.y;
  const R m1 = p1.x * p1.x + p1.y * p1.y;
  *e0 = k.kuu * m0 + k.kud * m1;
  *e1 = k.kdd * m1 + k.kud * m0;
}
template <typename R> __device__ __forceinline__ R larger(R a, R b) { return fmax(a, fabs(b)); }

// Code variants of the block. NT: no coupling phase (theta = 0).
enum { PV_REAL_SMALL, PV_REAL, PV_IMAG_SMALL_NT, PV_IMAG_SMALL, PV_IMAG };
template <int V> struct PointVariant { static constexpr int v = V; };

// Calls f(PointVariant<V>) for the variant of an instance; `top` is the
// largest phase of this thread's points. The choice is uniform over the wave.
// The theta-free variant is complex64's alone: there it saves 1-3 % of a batched
// row pass, in complex128 the third way out of the branch costs more registers
// than its arithmetic saves (32 x 256^2: 37.5 us with it, 32.3 without).
template <typename R, bool NT = sizeof(R) == 4, class F>
__device__ __forceinline__ void with_variant(const RowCoef<R>& k, R top, F&& f) {
  if (k.imag) {
    if (__builtin_amdgcn_ballot_w64(!(top <= (R)kSmallExp))) {
      f(PointVariant<PV_IMAG>());
    } else {
      if constexpr (NT) {
        if (!k.theta) return f(PointVariant<PV_IMAG_SMALL_NT>());
      }
      f(PointVariant<PV_IMAG_SMALL>());
    }
  } else if (__builtin_amdgcn_ballot_w64(!(top <= (R)kSmallAngle))) {
    f(PointVariant<PV_REAL>());
  } else {
    f(PointVariant<PV_REAL_SMALL>());
  }
}

// One point. FAST: separable potential (x and y tables tx, py) and uniform
// coupling factors; otherwise `a`, `b` are the point's coupling factors and
// f0, f1 its potential factors.
template <typename R, int V, typename C>
__device__ __forceinline__ void point_ops(C& p0, C& p1, R e0, R e1, R sc, R a, R b, C f0, C f1, C e) {
  constexpr bool IMAG = V >= PV_IMAG_SMALL_NT;
  constexpr bool SMALL = V != PV_REAL && V != PV_IMAG;
  constexpr bool NT = V == PV_IMAG_SMALL_NT;
  const C u0 = phase_op<R, IMAG, SMALL>(e0);
  const C u1 = phase_op<R, IMAG, SMALL>(e1);
  const R s = NT ? b : b * e.x, r = NT ? (R)0 : b * e.y;
  p0 = mul_phase<IMAG>(p0, u0);
  p1 = mul_phase<IMAG>(p1, u1);
  // First half of the coupling (tensor_propagator.py:252-254), scaled.
  mix<IMAG, NT>(p0, p1, a * sc, s * sc, NT ? (R)0 : r * sc);
  p0 = mul_phase<IMAG>(p0, f0);       // potential (:256)
  p1 = mul_phase<IMAG>(p1, f1);
  mix<IMAG, NT>(p0, p1, a, s, r);     // second half (:258-260)
  p0 = mul_phase<IMAG>(p0, u0);       // the same U again (:267)
  p1 = mul_phase<IMAG>(p1, u1);
}

// x times y factor of a potential phase (real in imaginary time).
template <bool IMAG, typename C> __device__ __forceinline__ C pot_factor(C tx, C py) {
  if constexpr (IMAG)
    return C{tx.x * py.x, 0};
  else
    return cmul(tx, py);
}

// The y factor of every point of one row.
template <typename C> struct RowFactor {
  C v;
  __device__ __forceinline__ C operator[](int) const { return v; }
};

// Offsets j T of a thread's points of a row.
template <int T> struct RowStride {
  __device__ __forceinline__ size_t operator()(int j) const { return (size_t)(j * T); }
};

// Points J0 <= j < J1 of a row on the fast operator path, in one variant. PY:
// the points' y factors (RowFactor, or one per point).
template <typename R, int V, int E, int J0, int J1, typename C, typename PY>
__device__ __forceinline__ void fast_points(C (&a0)[E], C (&a1)[E], const RowCoef<R>& k, const PY& py0, const PY& py1,
                                            const C (&tx0)[E], const C (&tx1)[E], const C (&tex)[E]) {
  constexpr bool IMAG = V >= PV_IMAG_SMALL_NT;
#pragma unroll
  for (int j = J0; j < J1; ++j) {
    R e0, e1;
    point_phases<R>(a0[j], a1[j], k, &e0, &e1);
    point_ops<R, V>(a0[j], a1[j], e0, e1, k.sc, k.ca, k.cb, pot_factor<IMAG>(tx0[j], py0[j]),
                    pot_factor<IMAG>(tx1[j], py1[j]), tex[j]);
  }
}

// Largest phase of the points J0 <= j < J1 (fast operator path).
template <typename R, int E, int J0, int J1, typename C>
__device__ __forceinline__ R fast_top(const C (&a0)[E], const C (&a1)[E], const RowCoef<R>& k) {
  R top = (R)0;
#pragma unroll
  for (int j = J0; j < J1; ++j) {
    R e0, e1;
    point_phases<R>(a0[j], a1[j], k, &e0, &e1);
    top = larger(larger(top, e0), e1);
  }
  return top;
}

// Points J0 <= j < J1 of a row: FAST as above, else with dense potentials and
// coupling arrays where the slot has them (point j at base + offset(j) of
// them). Their values are read inside the point loop: read ahead of the variant
// test, for a test that counts them too, they cost 10 to 30 registers, which is a
// wave per SIMD or a spill in most shapes. Row pass in imaginary time, dense
// potential and coupling, us, read ahead -> here: 2048 x 1024 complex128 62.4 ->
// 52.7, complex64 64.7 -> 43.9, 8 x 512^2 complex128 66.1 -> 57.6, complex64 35.4 ->
// 33.2, one 512^2 complex128 12.8 -> 12.4.
template <typename R, int E, bool FAST, int J0 = 0, int J1 = E, typename C, typename PY, typename At>
__device__ __forceinline__ void row_pointwise(C (&a0)[E], C (&a1)[E], const InstDev& P, const RowCoef<R>& k,
                                              size_t base, const At& offset, const PY& py0, const PY& py1, const C (&tx0)[E],
                                              const C (&tx1)[E], const C (&tex)[E]) {
  if constexpr (FAST) {
    with_variant<R>(k, fast_top<R, E, J0, J1>(a0, a1, k), [&](auto v) {
      fast_points<R, decltype(v)::v, E, J0, J1>(a0, a1, k, py0, py1, tx0, tx1, tex);
    });
  } else {
    const double* vd0 = P.v_dense[0];
    const double* vd1 = P.v_dense[1];
    const double* omd = P.coupling == 2 ? P.omega_dense : nullptr;
    // A slot whose dense phases are not all small takes the general code; the
    // interaction phases decide for the others.
    const R top = k.dense_small ? fast_top<R, E, J0, J1>(a0, a1, k) : (R)INFINITY;
    with_variant<R, false>(k, top, [&](auto v) {
      constexpr int V = decltype(v)::v;
      constexpr bool IMAG = V >= PV_IMAG_SMALL_NT;
      constexpr bool SMALL = V != PV_REAL && V != PV_IMAG;
#pragma unroll
      for (int j = J0; j < J1; ++j) {
        const size_t at = base + offset(j);
        R a = k.ca, b = k.cb;
        if (omd) {
          const R an = (R)ld_global(omd + at) * k.dts * (R)0.25;
          if constexpr (IMAG) {
            const R g = SMALL ? ex_poly(an) : ex<R>(an), gi = (R)1 / g;
            a = (R)0.5 * (g + gi);
            b = (R)-0.5 * (g - gi);
          } else {
            const C u = phase_op<R, false, SMALL>(an);
            a = u.x;
            b = u.y;
          }
        }
        const C f0 = vd0 ? phase_op<R, IMAG, SMALL>((R)ld_global(vd0 + at) * k.dts) : pot_factor<IMAG>(tx0[j], py0[j]);
        const C f1 = vd1 ? phase_op<R, IMAG, SMALL>((R)ld_global(vd1 + at) * k.dts) : pot_factor<IMAG>(tx1[j], py1[j]);
        R e0, e1;
        point_phases<R>(a0[j], a1[j], k, &e0, &e1);
        point_ops<R, V>(a0[j], a1[j], e0, e1, k.sc, a, b, f0, f1, tex[j]);
      }
    });
  }
}

// ---------------------------------------------------------------- row pass

// The x-table values (potential phases of both components, e^{-i theta})
// of this thread's points J0 <= j < J1 of a row; `stand_in` replaces an
// absent potential table. Global loads: issued before a transform's last
// LDS exchange, they stay in flight across its waits.
template <int E, int T, int J0 = 0, int J1 = E, typename C>
__device__ __forceinline__ void load_x_tables(C (&tx0)[E], C (&tx1)[E], C (&tex)[E], const C* px0, const C* px1,
                                              const C* eth, const C* stand_in, int t) {
  const C* s0 = px0 ? px0 : stand_in;
  const C* s1 = px1 ? px1 : stand_in;
#pragma unroll
  for (int j = J0; j < J1; ++j) {
    tx0[j] = ld_global(s0 + t + j * T);
    tx1[j] = ld_global(s1 + t + j * T);
    tex[j] = ld_global(eth + t + j * T);
  }
}

// The row pointwise block point by point from point J on, point J's tables
// already loaded: point J + 1's tables are loaded first, so their latency
// overlaps point J's arithmetic, and at most two points' tables are live.
// `point` is called with std::integral_constant-like PointVariant<J>.
template <int E, int T, int J, typename C, class F>
__device__ __forceinline__ void pointwise_points(int t, C (&tx0)[E], C (&tx1)[E], C (&tex)[E], const C* px0,
                                                 const C* px1, const C* eth, const C* tws, F&& point) {
  if constexpr (J < E) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (J + 1 < E) load_x_tables<E, T, J + 1, J + 2>(tx0, tx1, tex, px0, px1, eth, tws, t);
    point(PointVariant<J>());
    pointwise_points<E, T, J + 1>(t, tx0, tx1, tex, px0, px1, eth, tws, point);
  }
}

// Population record of one full step from the column pass's S sums
// (tensor_propagator.py:194): pops[2 (step - 1) + s] for step > 0 within
// the run's capacity. Every thread of the wave gets the sums; thread 0
// writes.
template <bool COH = false>
__device__ __forceinline__ void record_pops(const InstDev& P, double* pops, int cap, int step, int nt2) {
  const double* part = P.part;
  double ps[2] = {wave_sum_strided<COH>(part + PART_S * nt2, nt2 / 2),
                  wave_sum_strided<COH>(part + PART_S * nt2 + nt2 / 2, nt2 / 2)};
  if (threadIdx.x == 0 && step > 0 && pops && step - 1 < cap) {
    const double tot = ps[0] + ps[1];
    pops[2 * (step - 1) + 0] = P.atom_num * ps[0] / tot;
    pops[2 * (step - 1) + 1] = P.atom_num * ps[1] / tot;
  }
}

// One block of ROWS row pairs (both components) of one instance (the body of
// row_pass_kernel and of the persistent step kernel). `gate` is called once
// every global load of the prologue has been issued; false drops the block.
// GENERAL: some slot has a dense potential or a coupling array; otherwise
// every slot takes the separable fast path.
// HELD: see row_pass_kernel.
template <typename R, int N, int E, int ROWS, bool GENERAL, int CM, bool HELD = false, class Gate>
__device__ __forceinline__ void row_item(const InstDev& P, typename Cx<R>::T* __restrict__ psi, int ny,
                                         const double* __restrict__ part, const typename Cx<R>::T* __restrict__ tws,
                                         int dur, int col_w, int stream, int blk, double* smem, Gate gate) {
  typedef typename Cx<R>::T C;
  typedef SwzView<sizeof(C)> V;
  constexpr int T = N / E;
  // LDS: [ROWS*2*N exchange][N twiddles][ROWS*2*N second exchange buffer,
  // when double-buffered]. The x phase tables stay in global memory (cache
  // resident): copies in LDS would cost occupancy.
  constexpr size_t kData = (size_t)ROWS * 2 * N * sizeof(C);
  constexpr bool kTw = tw_in_lds(kData, N, sizeof(C));
  constexpr bool kDb = row_double_buffer(E, kData, kTw ? (size_t)N * sizeof(C) : 0);
  // A row's T threads are consecutive lanes: with T <= 64 each row's
  // transforms lie within one wave.
  constexpr bool kWave = T <= 64;
  const int nt2 = 2 * (N / col_w);
  const int row = threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int y = blk * ROWS + row;
  C* const sm = reinterpret_cast<C*>(smem);
  C* r0 = psi + (size_t)y * N;
  C* r1 = r0 + (size_t)ny * N;
  C* lds0 = sm + (size_t)row * 2 * N;
  C* lds1 = lds0 + N;

  // Global loads first: the norm partials, the two rows and the twiddles (held
  // in registers until they are stored to LDS); the kernel then waits for
  // memory once.
  const PartSum psum(part + PART_NRM * nt2, CM ? 0 : nt2);
  C a0[E], a1[E];
  // CM: as in col_item; element (comp, y, x) at byte ((comp ny + y) N + x) sizeof(C)
  const CoherentBuf cb(psi, CM ? (uint32_t)(2 * (size_t)ny * N * sizeof(C)) : 0u);
  const uint32_t c0 = (uint32_t)(((size_t)y * N + t) * sizeof(C));
  const uint32_t c1 = c0 + (uint32_t)((size_t)ny * N * sizeof(C));
  if constexpr ((CM & CM_LOAD) != 0) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      a0[j] = cb.load<C>(c0 + (uint32_t)(j * T * sizeof(C)));
      a1[j] = cb.load<C>(c1 + (uint32_t)(j * T * sizeof(C)));
    }
  } else if (stream) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      a0[j] = ld_stream(r0 + t + j * T);
      a1[j] = ld_stream(r1 + t + j * T);
    }
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      a0[j] = ld_global(r0 + t + j * T);
      a1[j] = ld_global(r1 + t + j * T);
    }
  }
  constexpr int kBlock = ROWS * T;
  const double* vd0 = P.v_dense[0];
  const double* vd1 = P.v_dense[1];
  C py0 = C{(R)1, (R)0}, py1 = C{(R)1, (R)0};
  const C* px0 = nullptr;
  const C* px1 = nullptr;
  if (!vd0) {
    py0 = ld_global(reinterpret_cast<const C*>(P.py[dur][0]) + y);
    px0 = reinterpret_cast<const C*>(P.px[dur][0]);
  }
  if (!vd1) {
    py1 = ld_global(reinterpret_cast<const C*>(P.py[dur][1]) + y);
    px1 = reinterpret_cast<const C*>(P.px[dur][1]);
  }
  const C* eth = reinterpret_cast<const C*>(P.etheta);
  constexpr bool kEarlyTables = E <= 2;
  C tx0[E], tx1[E], tex[E];
  if constexpr (kEarlyTables) load_x_tables<E, T>(tx0, tx1, tex, px0, px1, eth, tws, t);
  TableStage<kTw, N, kBlock, C> stw;
  stw.load(tws);
  if (!gate()) return;

  // Real-space normalization (tensor_tools.py:301-305) from the column
  // pass's k-space sums by Parseval: sum_r |IDFT2 v|^2 = Nx Ny sum_k |v|^2.
  // Every wave sums all partials itself (same order in every wave and
  // block: no barrier, deterministic), loaded ahead of the rows. The twiddles stored here are published by the transform's first barrier
  // (its first stage uses none).
  const double nrm = CM ? wave_sum_strided<(CM & CM_LOAD) != 0>(part + PART_NRM * nt2, nt2) : psum.sum();
  const C* tw = stw.store(sm + ROWS * 2 * N);
  if constexpr (kWave && kTw) __syncthreads();  // publishes the twiddles staged by every wave
  const double lam2 = P.atom_num / (P.dv_r * (double)N * (double)ny * nrm);

  C* const alt0 = sm + ROWS * 2 * N + (kTw ? N : 0) + (size_t)row * 2 * N;
  C* const alt1 = alt0 + N;
  if constexpr (kDb)
    fft_run2_db<N, E, true, V, kWave>(a0, a1, t, tw, lds0, lds1, alt0, alt1);
  else if constexpr (kTw) {
    fft_run2<N, E, true, V, kWave>(a0, a1, t, tw, lds0, lds1);
  } else {
    const StageTwiddles<N, E, 1, C> none{};
    fft_run2_pre<N, E, true, V, kWave>(a0, a1, t, tw, lds0, lds1, none);
  }

  // The x-table values of this thread's points (an absent potential table
  // is stood in for by the global twiddle table: N entries, unused). Radix
  // 2: loaded with the state at the start (few registers to hold them
  // through the inverse transform). Radix 4: after the inverse transform,
  // in two halves, the second loaded only after the first half of the
  // points is done (the scheduling barrier keeps the compiler from hoisting
  // those loads), so at most half of them are live at once: 216 -> 162
  // VGPRs for the complex128 pass (3 waves per SIMD instead of 2), paid for
  // with one more L2 round trip per row. Complex128 radix >= 8: point by
  // point, each point's tables loaded while the previous point is computed
  // (296 -> 224 VGPRs, 2 waves per SIMD; with the twiddles in global memory
  // two 2048-point workgroups share a CU). Complex64 radix >= 8 uses the
  // halves, which already fit 3 waves per SIMD (point by point would only
  // add latency).
  const RowCoef<R> k(P, dur, lam2);
  const RowFactor<C> fy0{py0}, fy1{py1};
  if constexpr (E >= 8 && sizeof(C) == 16) {
    load_x_tables<E, T, 0, 1>(tx0, tx1, tex, px0, px1, eth, tws, t);
    if constexpr (GENERAL)
      pointwise_points<E, T, 0>(t, tx0, tx1, tex, px0, px1, eth, tws, [&](auto j) {
        constexpr int J = decltype(j)::v;
        row_pointwise<R, E, false, J, J + 1>(a0, a1, P, k, (size_t)y * N + t, RowStride<T>(), fy0, fy1, tx0, tx1, tex);
      });
    else {
      const R top = fast_top<R, E, 0, E>(a0, a1, k);
      // Opaque copies: the densities are formed again point by point rather
      // than held for all points at once (32 registers, past 256).
#pragma unroll
      for (int j = 0; j < E; ++j)
        asm volatile("" : "+v"(a0[j].x), "+v"(a0[j].y), "+v"(a1[j].x), "+v"(a1[j].y));
      with_variant<R>(k, top, [&](auto v) {
        pointwise_points<E, T, 0>(t, tx0, tx1, tex, px0, px1, eth, tws, [&](auto j) {
          constexpr int J = decltype(j)::v;
          fast_points<R, decltype(v)::v, E, J, J + 1>(a0, a1, k, fy0, fy1, tx0, tx1, tex);
        });
      });
    }
  } else {
    constexpr int H = kEarlyTables ? E : E / 2;
    if constexpr (!kEarlyTables) load_x_tables<E, T, 0, H>(tx0, tx1, tex, px0, px1, eth, tws, t);
    row_pointwise<R, E, !GENERAL, 0, H>(a0, a1, P, k, (size_t)y * N + t, RowStride<T>(), fy0, fy1, tx0, tx1, tex);
    if constexpr (H < E) {
      __builtin_amdgcn_sched_barrier(0);
      load_x_tables<E, T, H, E>(tx0, tx1, tex, px0, px1, eth, tws, t);
      row_pointwise<R, E, !GENERAL, H, E>(a0, a1, P, k, (size_t)y * N + t, RowStride<T>(), fy0, fy1, tx0, tx1, tex);
    }
  }
  // Large rows: the forward transform and the stores index by an opaque copy
  // of t, so their LDS and state addresses are recomputed here instead of
  // being held in registers since the loads and the inverse transform, which
  // compute the same addresses (held, they cost up to 70 VGPRs and spill the
  // 4096-point complex128 pass). It pays where registers are what limits
  // the resident workgroups: 2048 points and more (complex64 2048 points: 192 ->
  // 130 VGPRs, 58 -> 50 us per pass; complex128, unless HELD: 98 -> 79 us for 2048
  // rows), and 1024 points where the LDS admits three waves per SIMD. With
  // small batched rows, whose workgroups fill the CUs' slots already, only the
  // recomputation remains (+2 %).
  constexpr size_t kLdsWg = kData * (kDb ? 2 : 1) + (kTw ? (size_t)N * sizeof(C) : 0);
  constexpr int kLdsWaves = (int)(kLdsBytes / kLdsWg) * ((ROWS * T + 63) / 64) / 4;
  constexpr bool kOpaque = HELD ? false : N >= 2048 || (N >= 1024 && kLdsWaves >= 3);
  int tf = t;
  if constexpr (kOpaque) asm volatile("" : "+v"(tf));
  // The forward transform starts on the buffer pair the inverse one read
  // last but one, so no barrier is needed between them.
  if constexpr (kDb && fft_exchanges<N, E>() % 2)
    fft_run2_db<N, E, false, V, kWave>(a0, a1, tf, tw, alt0, alt1, lds0, lds1);
  else if constexpr (kDb)
    fft_run2_db<N, E, false, V, kWave>(a0, a1, tf, tw, lds0, lds1, alt0, alt1);
  else if constexpr (kTw) {
    fft_run2<N, E, false, V, kWave>(a0, a1, tf, tw, lds0, lds1);
  } else {
    const StageTwiddles<N, E, 1, C> none{};
    fft_run2_pre<N, E, false, V, kWave>(a0, a1, tf, tw, lds0, lds1, none);
  }
  if constexpr ((CM & CM_STORE) != 0) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      cb.store<C>(c0 + (uint32_t)(j * T * sizeof(C)), a0[j]);
      cb.store<C>(c1 + (uint32_t)(j * T * sizeof(C)), a1[j]);
    }
  } else if (stream) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      st_stream(r0 + tf + j * T, a0[j]);
      st_stream(r1 + tf + j * T, a1[j]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      st_global(r0 + tf + j * T, a0[j]);
      st_global(r1 + tf + j * T, a1[j]);
    }
  }
}

// Waves per SIMD asked of the compiler: two for the complex128 radix >= 8 row
// passes whose LDS admits two (it would otherwise take 260-298 registers for
// some of them, which leaves one).
template <typename R, int N, int E, int ROWS> constexpr int row_min_waves() {
  constexpr size_t cs = sizeof(typename Cx<R>::T);
  constexpr size_t data = (size_t)ROWS * 2 * N * cs;
  constexpr size_t lds = data + (tw_in_lds(data, N, cs) ? (size_t)N * cs : 0);
  constexpr int waves = (int)(kLdsBytes / lds) * ((ROWS * (N / E) + 63) / 64) / 4;
  return E >= 8 && cs == 16 && waves >= 2 ? 2 : 1;
}

// HELD: for launches of at most one workgroup per CU (launch_row), where
// registers limit nothing: addresses and twiddles kept from the inverse
// transform to the forward one (at the price of a few spills). Complex128
// 2048-point rows, 256 of them: 21.3 us instead of 24.7; with 2048 of them it
// would be 98 instead of 79.
template <typename R, int N, int E> constexpr bool row_has_held() { return sizeof(R) == 8 && N == 2048 && E == 8; }
template <typename R, int N, int E, int ROWS, bool GENERAL, bool HELD = false>
__global__ __launch_bounds__(ROWS*(N / E), (row_min_waves<R, N, E, ROWS>())) void row_pass_kernel(const InstDev* __restrict__ insts,
                                                                RunDev* __restrict__ runs, void* direct_psi,
                                                                const double* direct_part, int direct_n,
                                                                const typename Cx<R>::T* __restrict__ tws,
                                                                int dur, int first_sub, int col_w, int stream) {
  typedef typename Cx<R>::T C;
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  RunDev& run = runs[inst];
  const InstDev& P = insts[inst];
  // Addresses of the state and the partial sums, and the column length: kernel
  // arguments for a single-slot plan (loads first, active flag checked after
  // them), else read together with the active flag (one round of scalar loads
  // before the state loads).
  const bool direct = direct_psi != nullptr;
  C* const psi = reinterpret_cast<C*>(direct ? direct_psi : P.psi);
  const int ny = direct ? direct_n : P.ny;
  if (!direct && (!run.active || !psi || ny <= 0)) return;
  auto gate = [&]() -> bool {
    if (direct) {
      // The prologue loads stay ahead of the flag test (a loaded slot's
      // state and tables stay allocated when it is inactive).
      asm volatile("" ::: "memory");
      if (!run.active) return false;
    }
    // Block 0 of the first sub-step records the previous full step's
    // populations and counts the step; the state leaves this pass in hybrid
    // form (no other block of this kernel reads the flag; the next column
    // pass does).
    if (blockIdx.x == 0) {
      if (first_sub) {
        const int step = run.step;
        record_pops(P, run.pops, run.pops_cap, step, 2 * (N / col_w));
        if (threadIdx.x == 0) run.step = step + 1;
      }
      if (threadIdx.x == 0) run.form = FORM_HYBRID;
    }
    return true;
  };
  row_item<R, N, E, ROWS, GENERAL, 0, HELD>(P, psi, ny, direct ? direct_part : P.part, tws, dur, col_w, stream, blockIdx.x, smem, gate);
}

// Row pass with the two components on separate waves (the split layout):
// ROWS rows per workgroup, each taken by two waves of T = N/E = 64 threads,
// wave c transforming component c with exchanges inside the wave (no
// workgroup barrier). The two waves meet in LDS for the pointwise block,
// which all 128 threads of the row share (N/128 points each), then each wave
// transforms its component back. Against the layout above (both components
// per thread, transforms spread over several waves) this halves the LDS
// exchanges per transform at 512 points: 10.7 vs 11.8 us per pass for one
// 512^2 complex128 instance, 9.2 vs 9.5 us in complex64 (same-host A/B). The
// tuner picks it per grid and batch size; rows per workgroup are encoded as
// -ROWS in the shape tables.
template <typename R, int N, int E, int ROWS, bool GENERAL>
__global__ __launch_bounds__(ROWS * 2 * (N / E)) void row_split_kernel(const InstDev* __restrict__ insts,
                                                                       RunDev* __restrict__ runs, void* direct_psi,
                                                                       const double* direct_part, int direct_n,
                                                                       const typename Cx<R>::T* __restrict__ tws,
                                                                       int dur, int first_sub, int col_w, int stream) {
  typedef typename Cx<R>::T C;
  typedef SwzView<sizeof(C)> V;
  constexpr int T = N / E;
  static_assert(T == 64, "one wave per component");
  constexpr int TP = 2 * T;   // threads of one row
  constexpr int EP = N / TP;  // pointwise points per thread
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  RunDev& run = runs[inst];
  const InstDev& P = insts[inst];
  // State address and column length as in row_pass_kernel.
  const bool direct = direct_psi != nullptr;
  C* const psi = reinterpret_cast<C*>(direct ? direct_psi : P.psi);
  const int ny = direct ? direct_n : P.ny;
  if (!direct && (!run.active || !psi || ny <= 0)) return;
  const int rw = threadIdx.x / TP;
  const int y = blockIdx.x * ROWS + rw;
  const int tid = threadIdx.x % TP;
  const int comp = tid / T;
  const int t = tid % T;
  // LDS: [ROWS][2][N] data (swizzled within each component), then the
  // twiddles when they fit (tw_in_lds).
  C* const sm = reinterpret_cast<C*>(smem) + rw * 2 * N;
  C* const lds = sm + comp * N;
  C* const row = psi + ((size_t)comp * ny + y) * N;
  constexpr size_t kData = (size_t)ROWS * 2 * N * sizeof(C);
  constexpr bool kTw = tw_in_lds(kData, N, sizeof(C));
  const int nt2 = 2 * (N / col_w);
  const PartSum psum((direct ? direct_part : P.part) + PART_NRM * nt2, nt2);  // ahead of the state, see PartSum
  C a[E];
  if (stream) {
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = ld_stream(row + t + j * T);
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = ld_global(row + t + j * T);
  }
  const double* vd0 = P.v_dense[0];
  const double* vd1 = P.v_dense[1];
  C py0 = C{(R)1, (R)0}, py1 = C{(R)1, (R)0};
  const C* px0 = nullptr;
  const C* px1 = nullptr;
  if (!vd0) {
    py0 = ld_global(reinterpret_cast<const C*>(P.py[dur][0]) + y);
    px0 = reinterpret_cast<const C*>(P.px[dur][0]);
  }
  if (!vd1) {
    py1 = ld_global(reinterpret_cast<const C*>(P.py[dur][1]) + y);
    px1 = reinterpret_cast<const C*>(P.px[dur][1]);
  }
  const C* eth = reinterpret_cast<const C*>(P.etheta);
  TableStage<kTw, N, ROWS * TP, C> stw;
  stw.load(tws);
  if (direct) {
    asm volatile("" ::: "memory");
    if (!run.active) return;
  }
  // Block 0 of the first sub-step records the previous full step's
  // populations and counts the step; the state leaves in hybrid form.
  if (blockIdx.x == 0) {
    if (first_sub) {
      const int step = run.step;
      record_pops(P, run.pops, run.pops_cap, step, nt2);
      if (threadIdx.x == 0) run.step = step + 1;
    }
    if (threadIdx.x == 0) run.form = FORM_HYBRID;
  }
  // Real-space normalization from the column pass's k-space sums (Parseval).
  const double nrm = psum.sum();
  const C* tw = stw.store(reinterpret_cast<C*>(smem) + ROWS * 2 * N);
  if constexpr (kTw) __syncthreads();  // publishes the twiddles to every wave
  const double lam2 = P.atom_num / (P.dv_r * (double)N * (double)ny * nrm);
  fft_run<N, E, true, V, true>(a, t, tw, lds);
  // The x tables of this thread's pointwise points, loaded here so that they
  // arrive while the workgroup meets at the barrier (loaded at the start,
  // they kept the prologue waiting for the slot descriptor's pointers).
  C tx0[EP], tx1[EP], tex[EP];
  load_x_tables<EP, TP>(tx0, tx1, tex, px0, px1, eth, tws, tid);
#pragma unroll
  for (int j = 0; j < E; ++j) lds[V::at(t + j * T)] = a[j];
  __syncthreads();
  C p0[EP], p1[EP];
#pragma unroll
  for (int j = 0; j < EP; ++j) {
    p0[j] = sm[V::at(tid + j * TP)];
    p1[j] = sm[N + V::at(tid + j * TP)];
  }
  const RowCoef<R> k(P, dur, lam2);
  row_pointwise<R, EP, !GENERAL>(p0, p1, P, k, (size_t)y * N + tid, RowStride<TP>(), RowFactor<C>{py0},
                                 RowFactor<C>{py1}, tx0, tx1, tex);
#pragma unroll
  for (int j = 0; j < EP; ++j) {
    sm[V::at(tid + j * TP)] = p0[j];
    sm[N + V::at(tid + j * TP)] = p1[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < E; ++j) a[j] = lds[V::at(t + j * T)];
  fft_run<N, E, false, V, true>(a, t, tw, lds);
  if (stream) {
#pragma unroll
    for (int j = 0; j < E; ++j) st_stream(row + t + j * T, a[j]);
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) st_global(row + t + j * T, a[j]);
  }
}

// --------------------------------------------------------------- normalize
// k-space renormalization to atom_num (tensor_propagator.py:271) from the
// exit column pass's S sums, plus the populations of the last step
// (tensor_propagator.py:194). Grid: (chunks, 1, n_inst).
template <typename R>
__global__ __launch_bounds__(256) void normalize_kernel(const InstDev* __restrict__ insts,
                                                        RunDev* __restrict__ runs, int col_w) {
  typedef typename Cx<R>::T C;
  __shared__ double scratch[16];
  const int inst = blockIdx.z;
  RunDev& run = runs[inst];
  if (!run.active) return;
  const InstDev& P = insts[inst];
  const int nt2 = 2 * (P.nx / col_w);
  double s[2];
  part_sums(P.part, nt2, PART_S, 1, s, scratch);
  const double tot = s[0] + s[1];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int step = run.step;
    if (step > 0 && run.pops && step - 1 < run.pops_cap) {
      run.pops[2 * (step - 1) + 0] = P.atom_num * s[0] / tot;
      run.pops[2 * (step - 1) + 1] = P.atom_num * s[1] / tot;
    }
  }
  const R kappa = (R)sqrt(P.atom_num / (P.dv_k * tot));
  C* psi = reinterpret_cast<C*>(P.psi);
  const size_t n = (size_t)2 * P.ny * P.nx;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    psi[i] = cscale(psi[i], kappa);
}

// Marks the state as normalized k-space. Separate launch so that no block of
// the normalize kernel can observe a half-updated flag.
static __global__ void set_form_kernel(RunDev* __restrict__ runs, int n, int form) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && runs[i].active) runs[i].form = form;
}

static __global__ void set_active_kernel(RunDev* __restrict__ runs, int slot, int active) {
  if (threadIdx.x == 0) runs[slot].active = active;
}

// Run-state (re)configuration for one slot; launched instead of copying so
// that it is ordered on the stream and graph-safe.
static __global__ void config_run_kernel(RunDev* __restrict__ runs, int slot, double* pops, int cap, int reset_step,
                                  int active, int form, double conv_tol) {
  if (threadIdx.x != 0) return;
  RunDev& r = runs[slot];
  r.pops = pops;
  r.pops_cap = cap;
  if (reset_step) {
    r.step = 0;
    r.converged = 0;
    r.n_checks = 0;
    r.e_prev = 0.0;
    r.steps_prev = 0;
  }
  if (active >= 0) r.active = active;
  if (form >= 0) r.form = form;
  r.conv_tol = conv_tol;
}

// ------------------------------------------------------------------ energy
// GP energy functional of a normalized k-space state, float64 sums:
//   E_kin = dv_k sum_s sum_k T_s |psik_s|^2
//   E_pot = dv_r sum_s sum_r V_s n_s, E_int = dv_r/2 sum (g_uu n0^2 + g_dd n1^2 + 2 g_ud n0 n1)
//   E_cpl = dv_r sum Omega Re(psi0* psi1 e^{-i theta}),  mu = (E_kin + E_pot + E_cpl + 2 E_int)/N
// with real space from chi = IDFT2(psik): n = |chi|^2 / (Nx Ny c)^2 (the
// (-1)^(x+y) of the shift cancels in every term). The transforms work in
// place: the column part leaves IDFT_y psik, the row part sums over
// IDFT_x IDFT_y psik and writes back DFT_x of it scaled by 1/(Nx Ny), and
// the restoring column part (FWD) applies DFT_y, which brings back psik up
// to rounding; no second copy of the state is needed.

// Column part: kinetic and norm sums in k-space, then IDFT_y in place; or
// (FWD) DFT_y in place, the last step of the evaluation.
template <typename R, int N, int E, int W, bool FWD>
__global__ __launch_bounds__(W*(N / E)) void energy_col_kernel(const InstDev* __restrict__ insts,
                                                               const RunDev* __restrict__ runs,
                                                               const typename Cx<R>::T* __restrict__ tws) {
  typedef typename Cx<R>::T C;
  typedef LdsView<W, 1 << 30, 0> V;
  constexpr int T = N / E;
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  if (!runs[inst].active) return;
  const InstDev& P = insts[inst];
  const int nx = P.nx;
  const int comp = blockIdx.y;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);  // neighbouring tiles share an L2
  const int c = threadIdx.x % W;
  const int t = threadIdx.x / W;
  const int jx = tile * W + c;
  C* lds = reinterpret_cast<C*>(smem) + c;
  C* col = reinterpret_cast<C*>(P.psi) + (size_t)comp * N * nx + jx;
  constexpr size_t kData = (size_t)W * N * sizeof(C);
  const C* tw = stage_twiddles<tw_in_lds(kData, N, sizeof(C))>(tws, N, reinterpret_cast<C*>(smem) + W * N);
  C a[E];
#pragma unroll
  for (int j = 0; j < E; ++j) a[j] = ld_global(col + (size_t)(t + j * T) * nx);
  if constexpr (FWD) {
    fft_run<N, E, false, V>(a, t, tw, lds);
#pragma unroll
    for (int j = 0; j < E; ++j) st_global(col + (size_t)(t + j * T) * nx, a[j]);
    return;
  }
  const double* td = P.t_dense[comp];
  const double tx = td ? 0.0 : P.tx[comp][jx];
  double kin = 0.0, s = 0.0;
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const int jy = t + j * T;
    const double tv = td ? td[(size_t)jy * nx + jx] : tx + P.ty[comp][jy];
    const double m = norm2d<R>(a[j]);
    kin += tv * m;
    s += m;
  }
  fft_run<N, E, true, V>(a, t, tw, lds);
#pragma unroll
  for (int j = 0; j < E; ++j) st_global(col + (size_t)(t + j * T) * nx, a[j]);
  double v[2] = {kin, s};
  block_sum<2>(v, smem);
  if (threadIdx.x == 0) {
    const int nt = nx / W;
    P.epart[EPART_KIN * P.estride + comp * nt + tile] = v[0];
    P.epart[EPART_S * P.estride + comp * nt + tile] = v[1];
  }
}

// Row part: IDFT_x of the rows, real-space sums, then DFT_x / (Nx Ny) in place.
template <typename R, int N, int E, int ROWS>
__global__ __launch_bounds__(ROWS*(N / E)) void energy_row_kernel(const InstDev* __restrict__ insts,
                                                                  const RunDev* __restrict__ runs,
                                                                  const typename Cx<R>::T* __restrict__ tws) {
  typedef typename Cx<R>::T C;
  typedef LdsView<1, 1 << 30, 0> V;
  constexpr int T = N / E;
  extern __shared__ double smem[];
  const int inst = blockIdx.z;
  if (!runs[inst].active) return;
  const InstDev& P = insts[inst];
  const int ny = P.ny;
  const int row = threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int y = blockIdx.x * ROWS + row;
  C* r0 = reinterpret_cast<C*>(P.psi) + (size_t)y * N;
  C* r1 = r0 + (size_t)ny * N;
  C* lds0 = reinterpret_cast<C*>(smem) + (size_t)row * 2 * N;
  C* lds1 = lds0 + N;
  constexpr size_t kData = (size_t)ROWS * 2 * N * sizeof(C);
  const C* tw = stage_twiddles<tw_in_lds(kData, N, sizeof(C))>(tws, N, reinterpret_cast<C*>(smem) + ROWS * 2 * N);
  C a0[E], a1[E];
#pragma unroll
  for (int j = 0; j < E; ++j) {
    a0[j] = ld_global(r0 + t + j * T);
    a1[j] = ld_global(r1 + t + j * T);
  }
  fft_run2<N, E, true, V>(a0, a1, t, tw, lds0, lds1);
  const double* vd0 = P.v_dense[0];
  const double* vd1 = P.v_dense[1];
  const double vy0 = vd0 ? 0.0 : P.vy[0][y];
  const double vy1 = vd1 ? 0.0 : P.vy[1][y];
  const C* eth = reinterpret_cast<const C*>(P.etheta);
  double pot = 0.0, inter = 0.0, cpl = 0.0, nrm = 0.0;
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const int x = t + j * T;
    const double m0 = norm2d<R>(a0[j]), m1 = norm2d<R>(a1[j]);
    const double v0 = vd0 ? vd0[(size_t)y * N + x] : P.vx[0][x] + vy0;
    const double v1 = vd1 ? vd1[(size_t)y * N + x] : P.vx[1][x] + vy1;
    pot += v0 * m0 + v1 * m1;
    inter += P.g_uu * m0 * m0 + P.g_dd * m1 * m1 + 2.0 * P.g_ud * m0 * m1;
    nrm += m0 + m1;
    if (P.coupling) {
      const double om = P.coupling == 2 ? P.omega_dense[(size_t)y * N + x] : P.omega;
      // Re(conj(a0) a1 e^{-i theta})
      double cr = (double)a0[j].x * a1[j].x + (double)a0[j].y * a1[j].y;
      double ci = (double)a0[j].x * a1[j].y - (double)a0[j].y * a1[j].x;
      if (eth) {
        const double er = (double)eth[x].x, ei = (double)eth[x].y;
        cr = cr * er - ci * ei;
      }
      cpl += om * cr;
    }
  }
  fft_run2<N, E, false, V>(a0, a1, t, tw, lds0, lds1);
  const R back = (R)(1.0 / ((double)N * (double)ny));
#pragma unroll
  for (int j = 0; j < E; ++j) {
    st_global(r0 + t + j * T, cscale(a0[j], back));
    st_global(r1 + t + j * T, cscale(a1[j], back));
  }
  double v[4] = {pot, inter, cpl, nrm};
  block_sum<4>(v, smem);
  if (threadIdx.x == 0) {
    P.epart[EPART_POT * P.estride + blockIdx.x] = v[0];
    P.epart[EPART_INT * P.estride + blockIdx.x] = v[1];
    P.epart[EPART_CPL * P.estride + blockIdx.x] = v[2];
    P.epart[EPART_NRM * P.estride + blockIdx.x] = v[3];
  }
}

// One block per slot: reduce the partials, write the energy terms and run
// the convergence test |E - E_prev| / |E| per full step <= conv_tol (a
// converged slot is deactivated, freezing its normalized k-space state).
static __global__ __launch_bounds__(256) void energy_final_kernel(const InstDev* __restrict__ insts,
                                                           RunDev* __restrict__ runs, int n_col_tiles,
                                                           int n_row_blocks, double* __restrict__ out) {
  __shared__ double scratch[32];
  const int inst = blockIdx.x;
  RunDev& run = runs[inst];
  if (!run.active) return;
  const InstDev& P = insts[inst];
  double v[6] = {0, 0, 0, 0, 0, 0};
  const int ncol = 2 * n_col_tiles;
  for (int i = threadIdx.x; i < ncol; i += blockDim.x) {
    v[0] += P.epart[EPART_KIN * P.estride + i];
    v[1] += P.epart[EPART_S * P.estride + i];
  }
  for (int i = threadIdx.x; i < n_row_blocks; i += blockDim.x) {
    v[2] += P.epart[EPART_POT * P.estride + i];
    v[3] += P.epart[EPART_INT * P.estride + i];
    v[4] += P.epart[EPART_CPL * P.estride + i];
    v[5] += P.epart[EPART_NRM * P.estride + i];
  }
  block_sum<6>(v, scratch);
  if (threadIdx.x != 0) return;
  const double kappa2 = P.atom_num / (P.dv_k * v[1]);
  const double nn = (double)P.nx * (double)P.ny * P.fft_c;
  const double a = kappa2 / (nn * nn);
  const double e_kin = kappa2 * P.dv_k * v[0];
  const double e_pot = P.dv_r * a * v[2];
  const double e_int = 0.5 * P.dv_r * a * a * v[3];
  const double e_cpl = P.dv_r * a * v[4];
  const double atoms = P.dv_r * a * v[5];
  const double e_tot = e_kin + e_pot + e_int + e_cpl;
  const double mu = (e_kin + e_pot + e_cpl + 2.0 * e_int) / atoms;
  double rel = -1.0;
  if (run.n_checks > 0) {
    const int steps = run.step - run.steps_prev;
    rel = fabs(e_tot - run.e_prev) / fabs(e_tot) / (double)(steps > 0 ? steps : 1);
    if (run.conv_tol > 0.0 && steps > 0 && rel <= run.conv_tol) {
      run.converged = 1;
      run.active = 0;
    }
  }
  const double e[8] = {e_tot, e_kin, e_pot, e_int, e_cpl, mu, atoms, rel};
  for (int i = 0; i < 8; ++i) {
    run.energy[i] = e[i];
    if (out) out[8 * inst + i] = e[i];
  }
  run.e_prev = e_tot;
  run.steps_prev = run.step;
  run.n_checks += 1;
}

// ------------------------------------------------- standalone primitives
// Device forms of tensor_tools.fft_2d / ifft_2d (tensor_tools.py:201-258):
//   fft_2d : fftshift(FFTN(psi)) * c  = DFT_y DFT_x [(-1)^(x+y) c psi]
//   ifft_2d: IFFTN(ifftshift(psik))/c = (-1)^(x+y) / (Nx Ny c) IDFT_x IDFT_y psik
// Both kernels transform up to two arrays per launch (the two spinor
// components), array blockIdx.z of the pair.
// Rows: optional pre- (forward) or post- (inverse) factor (-1)^(x+y) * scale.
template <typename R, int N, int E, int ROWS>
__global__ __launch_bounds__(ROWS*(N / E)) void fft_rows_kernel(FftPair io, int inv, int shift, double scale,
                                                                const typename Cx<R>::T* __restrict__ tws) {
  typedef typename Cx<R>::T C;
  typedef LdsView<1, 1 << 30, 0> V;
  constexpr int T = N / E;
  extern __shared__ double smem[];
  const int row = threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int y = blockIdx.x * ROWS + row;
  const C* src = reinterpret_cast<const C*>(io.in[blockIdx.z]) + (size_t)y * N;
  C* dst = reinterpret_cast<C*>(io.out[blockIdx.z]) + (size_t)y * N;
  C* lds = reinterpret_cast<C*>(smem) + (size_t)row * N;
  constexpr size_t kData = (size_t)ROWS * N * sizeof(C);
  const C* tw = stage_twiddles<tw_in_lds(kData, N, sizeof(C))>(tws, N, reinterpret_cast<C*>(smem) + ROWS * N);
  C a[E];
#pragma unroll
  for (int j = 0; j < E; ++j) a[j] = ld_global(src + t + j * T);
  // (-1)^(x+y) with x = t + j*T: T is even, so the sign depends on t and y only.
  const R f = (R)(shift && ((t + y) & 1) ? -scale : scale);
  if (!inv) {
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = cscale(a[j], f);
    fft_run<N, E, false, V>(a, t, tw, lds);
  } else {
    fft_run<N, E, true, V>(a, t, tw, lds);
#pragma unroll
    for (int j = 0; j < E; ++j) a[j] = cscale(a[j], f);
  }
  // Store addresses from an opaque copy of t: recomputed here rather than
  // held in registers since the loads (as in the pass kernels).
  int tf = t;
  asm volatile("" : "+v"(tf));
#pragma unroll
  for (int j = 0; j < E; ++j) st_global(dst + tf + j * T, a[j]);
}

template <typename R, int N, int E, int W>
__global__ __launch_bounds__(W*(N / E)) void fft_cols_kernel(FftPair io, int nx, int inv,
                                                             const typename Cx<R>::T* __restrict__ tws) {
  typedef typename Cx<R>::T C;
  typedef LdsView<W, 1 << 30, 0> V;
  constexpr int T = N / E;
  extern __shared__ double smem[];
  const C* in = reinterpret_cast<const C*>(io.in[blockIdx.z]);
  C* out = reinterpret_cast<C*>(io.out[blockIdx.z]);
  const int c = threadIdx.x % W;
  const int t = threadIdx.x / W;
  const int jx = xcd_tile(blockIdx.x, gridDim.x) * W + c;  // neighbouring tiles share an L2
  C* lds = reinterpret_cast<C*>(smem) + c;
  constexpr size_t kData = (size_t)W * N * sizeof(C);
  const C* tw = stage_twiddles<tw_in_lds(kData, N, sizeof(C))>(tws, N, reinterpret_cast<C*>(smem) + W * N);
  C a[E];
#pragma unroll
  for (int j = 0; j < E; ++j) a[j] = ld_global(in + (size_t)(t + j * T) * nx + jx);
  if (inv)
    fft_run<N, E, true, V>(a, t, tw, lds);
  else
    fft_run<N, E, false, V>(a, t, tw, lds);
  // Store addresses from an opaque copy of t (complex64 2048-point columns:
  // 84 -> 60 VGPRs, room for a second 1024-thread workgroup per CU).
  int tf = t;
  asm volatile("" : "+v"(tf));
#pragma unroll
  for (int j = 0; j < E; ++j) st_global(out + (size_t)(tf + j * T) * nx + jx, a[j]);
}

// Per-block sums of |psi0|^2 and |psi1|^2 (float64), written to part[2*block + s].
template <typename R>
__global__ __launch_bounds__(256) void density_sums_kernel(const typename Cx<R>::T* __restrict__ p0,
                                                           const typename Cx<R>::T* __restrict__ p1,
                                                           size_t n, double* __restrict__ part) {
  __shared__ double scratch[16];
  double v[2] = {0.0, 0.0};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    v[0] += norm2d<R>(p0[i]);
    v[1] += norm2d<R>(p1[i]);
  }
  block_sum<2>(v, scratch);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x + 0] = v[0];
    part[2 * blockIdx.x + 1] = v[1];
  }
}

// norm() (tensor_tools.py:261-311): nf = sum(dens0 + dens1) * vol / atom_num;
// out = psi / sqrt(nf); dens = |psi|^2 / nf. Every block reduces the same
// partials in the same order, so all blocks use the same nf. out may be psi
// (each element is read before it is written by the same thread); writing
// elsewhere saves the caller a copy of the state first. Bound by memory: 1024^2
// complex128 13.5 us out of place (80 MiB moved, 6.2 TB/s), 13.3 us in place
// behind two copies of 6.8 us; the call with its populations 76.1 -> 57.2 us.
template <typename R>
__global__ __launch_bounds__(256) void norm_apply_kernel(const typename Cx<R>::T* p0, const typename Cx<R>::T* p1,
                                                         size_t n, const double* __restrict__ part, int nblk,
                                                         double vol, double atom_num, typename Cx<R>::T* q0,
                                                         typename Cx<R>::T* q1, R* __restrict__ d0,
                                                         R* __restrict__ d1, double* __restrict__ nf_out) {
  __shared__ double scratch[16];
  double v[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < nblk; i += blockDim.x) v[0] += part[2 * i] + part[2 * i + 1];
  block_sum<2>(v, scratch);
  const double nf = v[0] * vol / atom_num;
  if (nf_out && blockIdx.x == 0 && threadIdx.x == 0) *nf_out = nf;
  const R inv_sqrt = (R)(1.0 / sqrt(nf));
  const R inv_nf = (R)(1.0 / nf);
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const typename Cx<R>::T a = p0[i], b = p1[i];
    if (d0) d0[i] = (R)((a.x * a.x + a.y * a.y) * inv_nf);
    if (d1) d1[i] = (R)((b.x * b.x + b.y * b.y) * inv_nf);
    q0[i] = cscale(a, inv_sqrt);
    q1[i] = cscale(b, inv_sqrt);
  }
}

// Final reduction of density_sums partials into out2[s] = vol * sum |psi_s|^2.
static __global__ __launch_bounds__(256) void pops_final_kernel(const double* __restrict__ part, int nblk, double vol,
                                                         double* __restrict__ out2) {
  __shared__ double scratch[16];
  double v[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < nblk; i += blockDim.x) {
    v[0] += part[2 * i];
    v[1] += part[2 * i + 1];
  }
  block_sum<2>(v, scratch);
  if (threadIdx.x == 0) {
    out2[0] = v[0] * vol;
    out2[1] = v[1] * vol;
  }
}

}  // namespace sgpe
