// Fused stage kernels of the OT potential and the split-operator step, on the
// register-resident line transforms of rfft.hpp.
//
// Every z pass works on pairs of adjacent z lines (x, 2p) and (x, 2p+1),
// contiguous in memory and packed as one complex line a + ib.  TPL lanes of
// one wavefront hold a pair, E points each (z = t + TPL*i), so the pointwise
// stages run in registers as the prologue or epilogue of the z transforms,
// field by field: a stage that consumes several spectra transforms them one
// after another and accumulates; a stage that produces several transforms and
// stores each as soon as it is formed.  Stencils in x and y read neighbouring
// lines from global memory (L2/MALL resident: adjacent planes are processed
// together).
//
//   zA    psi -> rho (stored) and, with backflow, q_d = rho v_d, q4 = rho |v|^2;
//         z r2c of {rho, q_x, q_y, q_z, q4} (and of rho~ = G rho, with rho~ in
//         place of rho in q_d and q4, under the HD / HD2 backflow switch)
//   xconv x forward FFT, k-space products with real kernel spectra and sums
//         over terms, x inverse FFT (a small program of outputs)
//   zAB   z c2r of {U*rho, U*q_d, U*q4} -> BF real part, W_d, BF imaginary part;
//         z c2r of Pi*rho -> local terms, Q, z r2c of Q;
//         z c2r of F*rho -> rho_st, G_d, z r2c of G_d
//   zBC   z c2r of J_d -> J_x, J_y (stored), H, KC term 3 and the z part of
//         term 1, BF divergence; z r2c of H
//   zC    x and y parts of KC term 1; z c2r of the summed linear terms; V += (API), or phase = e^{-iV dt/2}
//         and the first z pass of the propagator (step)
#pragma once
#include "fft_kernels.hpp"
#include "ot_common.hpp"

namespace dft {
namespace fused {

using rf::ColCfg;
using rf::LineCfg;
using rf::RP;

struct Ptrs8 {
  void *p[8];
};

// Addresses of a pair's points and of their periodic neighbours.  Line a is
// (ix, j), line b is (ix, j + 1); thread t holds points z = t + TPL*i of both.
// Every access is (element index of point t of some line) + a constant delta,
// so all points of a thread share a handful of per-thread offsets.
template <typename T, int N, int TPL> struct PairPos {
  uint32_t a0;         // point t of line a (line b is a0 + N)
  uint32_t xp0, xm0;   // point t of lines (ix +- 1, j)
  uint32_t ym0, yp1;   // point t of lines (ix, j - 1) and (ix, j + 2)
  int t;
  PairPos() = default;
  __device__ PairPos(uint32_t p, int t_, int nx, int ny) : t(t_) {
    const uint32_t l = 2 * p;
    const int j = (int)(l & (uint32_t)(ny - 1)), ix = (int)(l >> __builtin_ctz(ny));
    a0 = l * N + t;
    xp0 = ((uint32_t)((ix + 1) & (nx - 1)) * ny + j) * N + t;
    xm0 = ((uint32_t)((ix - 1) & (nx - 1)) * ny + j) * N + t;
    ym0 = ((uint32_t)ix * ny + ((j - 1) & (ny - 1))) * N + t;
    yp1 = ((uint32_t)ix * ny + ((j + 2) & (ny - 1))) * N + t;
  }
  static constexpr int kTPL = TPL;
  static constexpr int d(int w, int i) { return w * N + TPL * i; }
  // The same positions with offsets that the loads of the current stage
  // depend on (see rf::opaque_zero).
  __device__ PairPos here() const {
    PairPos r = *this;
    const uint32_t z = rf::opaque_zero();
    r.a0 += z;
    r.xp0 += z;
    r.xm0 += z;
    r.ym0 += z;
    r.yp1 += z;
    return r;
  }
  // field value at point (w, i)
  template <typename X> __device__ X at(const void *f, int w, int i) const { return rf::lde<X>(f, a0, d(w, i)); }
  // the same for a field this kernel reads only here
  template <typename X> __device__ X at_once(const void *f, int w, int i) const {
    return rf::lde_once<X>(f, a0, d(w, i));
  }
  template <typename X> __device__ void put(void *f, int w, int i, X v) const { rf::ste<X>(f, a0, v, d(w, i)); }
  // neighbour of point (w, i) one step along axis D in direction S (+1 / -1)
  template <typename X, int D, int S> __device__ X nb(const void *f, int w, int i) const {
    constexpr int E = N / TPL;
    if constexpr (D == 0) {
      return rf::lde<X>(f, S > 0 ? xp0 : xm0, d(w, i));
    } else if constexpr (D == 1) {
      if (S > 0) return w ? rf::lde<X>(f, yp1, TPL * i) : rf::lde<X>(f, a0, d(1, i));
      return w ? rf::lde<X>(f, a0, d(0, i)) : rf::lde<X>(f, ym0, TPL * i);
    } else {
      // z +- 1; only the last point of the line wraps forward, the first backward
      if (S > 0) {
        if (i < E - 1) return rf::lde<X>(f, a0, d(w, i) + 1);
        return rf::lde<X>(f, t == TPL - 1 ? a0 - t : a0 + TPL * i + 1, w * N);
      }
      if (i > 0) return rf::lde<X>(f, a0, d(w, i) - 1);
      return rf::lde<X>(f, t == 0 ? a0 + (N - 1) : a0 - 1, w * N);
    }
  }
};

// v_d = Im(psi* (psi_{+d} - psi_{-d})/2h) / (M (rho + eps)), clamped when
// enabled; f = 1 / (M (rho + eps)) is computed once per point for all axes.
template <typename T> __device__ __forceinline__ T velocity_factor(const PW<T> &pw, T r) {
  return pw.invM / (r + pw.eps_v);
}
// the same from psi at the point (s) and at its two neighbours (a: +d, b: -d)
template <typename T>
__device__ __forceinline__ T velocity_sab(const PW<T> &pw, T f, cplx<T> s, cplx<T> a, cplx<T> b) {
  const T dx = (a.x - b.x) * pw.inv2h, dy = (a.y - b.y) * pw.inv2h;
  T v = (s.x * dy - s.y * dx) * f;
  if (pw.clamp_v) v = clampv(v, pw.vmax);
  return v;
}
// Pair kernels use the plan with the fewest points per thread, 4: a line is
// one wavefront up to N = 256 and two at N = 512 (exchanges then take the
// block barrier).
template <int N> constexpr int pair_em() { return 4; }
template <int N>
using PairSync = std::conditional_t<(rf::RP<N, pair_em<N>()>::TPL <= 64), rf::WaveSync, rf::LineBlockSync>;

// Threads per block of the pair kernels.
template <typename T, int N> constexpr int PairBS = LineCfg<T, N, pair_em<N>()>::BS;

// Common prologue of the pair kernels.
#define FUSED_PAIR_SETUP()                                                   \
  using C = cplx<T>;                                                         \
  using G = LineCfg<T, N, pair_em<N>()>;                                     \
  constexpr int E = G::E, TPL = G::TPL, LP = G::LP;                          \
  __shared__ C s_x[G::LINES * LP];                                           \
  __shared__ C s_tw[rf::tw_len<T, N>()];                                     \
  const int ln = threadIdx.x / TPL, t = threadIdx.x % TPL;                   \
  const uint32_t p0 = (uint32_t)blockIdx.x * G::LINES + ln;                  \
  const bool act = p0 < npairs;                                              \
  /* out-of-range lanes compute on pair 0 and store nothing */               \
  const uint32_t p = act ? p0 : 0;                                           \
  C *X = s_x + ln * LP;                                                      \
  rf::load_tw<T, N, G::EM, G::BS>(s_tw, g_tw);                                 \
  __syncthreads();                                                           \
  const PairPos<T, N, TPL> q(p, t, pw.nx, pw.ny)

template <typename T> __device__ __forceinline__ T dens_of(cplx<T> s) { return s.x * s.x + s.y * s.y; }

// Neighbours a (+) and b (-) along axis D of the kept values s of a pair (X: real
// or complex).  Along y, line b is line a's neighbour and the other way round;
// along z the neighbours are other lanes' values (lines within a wavefront):
// point t + TPL i has z + 1 at lane t + 1 (index i), or at lane 0 (index i + 1)
// for t = TPL - 1, z - 1 likewise, wrapping around the line.  Only x, and one
// line each way along y, are loaded.
__device__ __forceinline__ float lane_of(float x, int l, int w) { return __shfl(x, l, w); }
__device__ __forceinline__ double lane_of(double x, int l, int w) { return __shfl(x, l, w); }
__device__ __forceinline__ float2 lane_of(float2 x, int l, int w) { return make_float2(__shfl(x.x, l, w), __shfl(x.y, l, w)); }
__device__ __forceinline__ double2 lane_of(double2 x, int l, int w) { return make_double2(__shfl(x.x, l, w), __shfl(x.y, l, w)); }
template <int D, class X, class Q, int E>
__device__ __forceinline__ void neighbours(const void *f, const Q &q, const X (&s)[2][E], int w, X (&a)[E], X (&b)[E]) {
  constexpr int TPL = Q::kTPL;
  if constexpr (D == 2 && TPL <= 64) {
    const int up = (q.t + 1) & (TPL - 1), dn = (q.t + TPL - 1) & (TPL - 1);
    X su[E], sd[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      su[i] = lane_of(s[w][i], up, TPL);
      sd[i] = lane_of(s[w][i], dn, TPL);
    }
#pragma unroll
    for (int i = 0; i < E; ++i) {
      a[i] = q.t == TPL - 1 ? su[(i + 1) % E] : su[i];
      b[i] = q.t == 0 ? sd[(i + E - 1) % E] : sd[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      a[i] = D == 1 && w == 0 ? s[1][i] : q.template nb<X, D, 1>(f, w, i);
      b[i] = D == 1 && w == 1 ? s[0][i] : q.template nb<X, D, -1>(f, w, i);
    }
  }
}

// Computes x here: arithmetic on registers whose result is needed only after
// later stages is otherwise sunk past their branches, with its operands (the
// loaded stencils) kept live in its place.
template <typename T> __device__ __forceinline__ void settle(T &x) { asm volatile("" : "+v"(x)); }

// r2c of the pair held in v and store of both half spectra to field `out`.
template <typename T, int N>
__device__ __forceinline__ void r2c_store(rf::Regs<T, N, pair_em<N>()> &v, cplx<T> *X, const cplx<T> *tw, int t,
                                          void *out, uint32_t p, int P, bool act) {
  rf::rfft<T, N, pair_em<N>(), -1, PairSync<N>>(v, X, tw, t);
  fft::split_store<T, N, pair_em<N>(), PairSync<N>>(v, X, t, out, p, P, act);
}

// Load + c2r of both lines of the pair from half-spectrum field `in`.
template <typename T, int N>
__device__ __forceinline__ void load_c2r(rf::Regs<T, N, pair_em<N>()> &v, cplx<T> *X, const cplx<T> *tw, int t,
                                         const void *in, uint32_t p, int P) {
  fft::load_merge<T, N, pair_em<N>()>(v, in, p, P, t);
  rf::rfft<T, N, pair_em<N>(), +1, PairSync<N>>(v, X, tw, t);
}

template <typename C> __device__ __forceinline__ auto &part(C &c, int w) { return w ? c.y : c.x; }

// -------------------------------------------------------------------- zA --
// Bound by the stores (psi in once, rho and five spectra out) and the loads of
// the psi stencils: with psi of the points kept and the y neighbours taken from
// the other line, 2.5 loads of psi per point instead of 5, zA 252 -> 214 us at
// 256^3 FP64 (192 -> 161 VGPRs, 3 waves per SIMD), 131 -> 129 FP32.
// HB: the backflow density switch of HD / HD2 (q_d = rho~ v_d, q4 = rho~ |v|^2
// and a sixth output, the transform of rho~ = G rho)
template <typename T, int N, bool BF, bool HB>
__device__ __forceinline__ void zA_body(const cplx<T> *psi, T *rho, Ptrs8 outs, int64_t npairs, int P, PW<T> pw,
                                        const cplx<T> *__restrict__ g_tw) {
  FUSED_PAIR_SETUP();
  // with backflow, psi of the points is kept for the three axes and q4
  C v[E], sp[2][E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
#pragma unroll
    for (int w = 0; w < 2; ++w) sp[w][i] = q.template at<C>(psi, w, i);
    v[i] = cmk<C>(dens_of<T>(sp[0][i]), dens_of<T>(sp[1][i]));
  }
  if (act) {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      q.template put<T>(rho, 0, i, v[i].x);
      q.template put<T>(rho, 1, i, v[i].y);
    }
  }
  if constexpr (BF) {
    // velocity factor per point, kept for the three axes
    T fv[2][E];
    T rt[2][HB ? E : 1];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      fv[0][i] = velocity_factor(pw, v[i].x);
      fv[1][i] = velocity_factor(pw, v[i].y);
      if constexpr (HB) {
        rt[0][i] = bf_rt(v[i].x, pw);
        rt[1][i] = bf_rt(v[i].y, pw);
        settle(rt[0][i]), settle(rt[1][i]);
      }
      settle(fv[0][i]), settle(fv[1][i]);
    }
    r2c_store<T, N>(v, X, s_tw, t, outs.p[0], p, P, act);
    T v2[2][E];
#pragma unroll
    for (int i = 0; i < E; ++i) v2[0][i] = v2[1][i] = 0;
    auto qd = [&](auto dtag) {
      constexpr int D = decltype(dtag)::value;
      T vr[2][E];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        C na[E], nb[E];
        neighbours<D>(psi, q.here(), sp, w, na, nb);
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const T vd = velocity_sab(pw, fv[w][i], sp[w][i], na[i], nb[i]);
          v2[w][i] += vd * vd;
          vr[w][i] = vd * (HB ? rt[w][HB ? i : 0] : dens_of<T>(sp[w][i]));
        }
      }
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = cmk<C>(vr[0][i], vr[1][i]);
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int i = 0; i < E; ++i) settle(v2[w][i]);
      r2c_store<T, N>(v, X, s_tw, t, outs.p[1 + D], p, P, act);
    };
    qd(std::integral_constant<int, 0>{});
    qd(std::integral_constant<int, 1>{});
    qd(std::integral_constant<int, 2>{});
#pragma unroll
    for (int i = 0; i < E; ++i) {
      if constexpr (HB) v[i] = cmk<C>(v2[0][i] * rt[0][i], v2[1][i] * rt[1][i]);
      else v[i] = cmk<C>(v2[0][i] * dens_of<T>(sp[0][i]), v2[1][i] * dens_of<T>(sp[1][i]));
    }
    r2c_store<T, N>(v, X, s_tw, t, outs.p[4], p, P, act);
    if constexpr (HB) {
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = cmk<C>(rt[0][i], rt[1][i]);
      r2c_store<T, N>(v, X, s_tw, t, outs.p[5], p, P, act);
    }
  } else {
    r2c_store<T, N>(v, X, s_tw, t, outs.p[0], p, P, act);
  }
}
template <typename T, int N, bool BF>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zA(const cplx<T> *psi, T *rho, Ptrs8 outs, int64_t npairs, int P, PW<T> pw,
         const cplx<T> *__restrict__ g_tw) {
  zA_body<T, N, BF, false>(psi, rho, outs, npairs, P, pw, g_tw);
}
template <typename T, int N>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zA_bfhd(const cplx<T> *psi, T *rho, Ptrs8 outs, int64_t npairs, int P, PW<T> pw,
              const cplx<T> *__restrict__ g_tw) {
  zA_body<T, N, true, true>(psi, rho, outs, npairs, P, pw, g_tw);
}

// ------------------------------------------------------------------ xconv --
struct MidTerm {
  int in, kern;  // of MidProg::in, MidProg::kern
  double scale;
};
struct MidOut {
  int nterms;
  MidTerm t[4];
  void *out;
};
constexpr int kMidMaxIn = 6, kMidMaxOut = 8, kMidMaxKern = 4;
struct MidProg {
  int nin, nout, nkern;
  const void *in[kMidMaxIn];
  MidOut o[kMidMaxOut];
  const void *kern[kMidMaxKern];  // the distinct kernel spectra the terms use
};

// What a launch of k_xconv reads of a program, as kernel arguments: single-term
// outputs (XOnes), or one output with several terms (XSum).  Arguments are fetched
// when a block starts, so it finds all it needs in one or two cache lines of them
// (us with the whole program, 0.75 KB, and with these: FP32 64^3 single-term output
// 5.9 and 5.3, sum 8.3 and 7.8; FP64 32^3 4.3 and 3.9, 6.8 and 6.1).
struct XOnes {
  struct {
    const void *in, *kern;
    void *out;
    double scale;
  } o[kMidMaxOut];
};
struct XSum {
  void *out;
  int nterms;
  struct {
    const void *in, *kern;
    double scale;
  } t[4];
};

// Blocks of the x-middle pass: ny * ntile tiles of COLS consecutive kz < P-1
// at one ky, and ceil(ny / COLS) tiles of the Nyquist column kz = P-1 over COLS
// consecutive ky.  A Nyquist tile touches one value per row, a cache line per
// lane, and takes several times as long as the others: these tiles go first,
// dealt over the XCDs by the plain block order, so that they overlap the rest
// instead of ending the launch alone (last, at 256^3 FP32: single-term outputs
// 305 us, accumulating 141; first: 252, 105).
template <int COLS> __host__ __device__ inline int mid_tiles(int P) { return (P - 1 + COLS - 1) / COLS; }
template <int COLS> __host__ __device__ inline int mid_blocks(int ny, int P) {
  return ny * mid_tiles<COLS>(P) + (ny + COLS - 1) / COLS;
}
// Output m (of nl) and column of lane `col` of this block, for a grid of
// mid_blocks * nl blocks.  Past the Nyquist tiles, consecutive logical blocks
// (the outputs of a tile, the tiles of one ky) are on one XCD, back to back.
struct MidCol {
  int m, o, kz;
  bool act;  // out-of-range lanes read an in-range column and store nothing
};
template <int COLS> __device__ __forceinline__ MidCol mid_col(int ny, int P, int nl, int col) {
  const int nyq = (ny + COLS - 1) / COLS * nl, ntile = mid_tiles<COLS>(P);
  int i = blockIdx.x;
  if (i < nyq) {
    const int t = i / nl, r = t * COLS + col;
    return {i - t * nl, r < ny ? r : ny - 1, P - 1, r < ny};
  }
  i -= nyq;
  const int n = ny * ntile * nl;
  const int L = (n & 7) == 0 ? (i & 7) * (n >> 3) + (i >> 3) : i, b = L / nl;
  const int o = b / ntile, c = (b - o * ntile) * COLS + col;
  return {L - b * nl, o, c < P - 1 ? c : P - 2, c < P - 1};
}

// Spectra are [nx][ny][PP] (P values per row) after the y pass; the x line
// (ky = o, kz) has stride ny*PP.  The arguments are indexed uniformly over the
// block (scalar loads); one output per block:
// out_m = F_x^-1 sum_t c_t F_x in_t over the terms of output m.  An input shared by
// several outputs is read once per output; the outputs of one column tile are
// consecutive logical blocks on one XCD, so those re-reads mostly hit that XCD's
// L2.  Bound by the movement of the x columns: without the transform the
// single-term FP32 outputs take 29 us per launch for 31 at 128^3, 170 for 183 at
// 256^3, 1565 for 1593 at 512^3 (profiler's times).  A block holds its lines, up
// to 16 points per thread: 4 waves per SIMD at 256 points FP32; the
// accumulating form adds an accumulator and the next term and runs at 2.
// Single-term outputs take 32 columns per block (256-byte row segments in FP32),
// the accumulating form 16.
// DFT_XCONV1_EM / DFT_XCONV1_COLS set that geometry for the single-term form,
// DFT_XCONV_EM / DFT_XCONV_COLS for the accumulating one; DFT_XCONV_MINB asks
// the register allocator for that many waves per SIMD (0: no request).
// Without the next-term prefetch below, 4 fit the accumulating form in 128
// VGPRs with 60 bytes per lane of spills: 165 -> 144 us at 256^3 FP32 (152
// VGPRs, 3 waves, without the request); with the prefetch, 2.
#ifndef DFT_XCONV1_EM
#define DFT_XCONV1_EM 16
#endif
#ifndef DFT_XCONV1_COLS
#define DFT_XCONV1_COLS 32
#endif
#ifndef DFT_XCONV_EM
#define DFT_XCONV_EM 16
#endif
#ifndef DFT_XCONV_COLS
#define DFT_XCONV_COLS 16
#endif
#ifndef DFT_XCONV_MINB
#define DFT_XCONV_MINB 2
#endif
// FP32 accumulating outputs read the next term's input and kernel before the
// current term's transform (+32 VGPRs: with it they run at 2 waves per SIMD
// without spills, 146 -> 139 us at 256^3; at 3 they spill and take 161 us)
#ifndef DFT_XCONV_PF
#define DFT_XCONV_PF 1
#endif
// the same request for the FP64 instantiations (0: none)
#ifndef DFT_XCONV_MINB64
#define DFT_XCONV_MINB64 2
#endif
// (N = 512 takes 8 columns: 45 KB of LDS in FP32 and 80
// in FP64, so that 3 or 2 blocks share a CU and one's barriers overlap another's
// loads; 16 columns fill it with one.  512^3 FP32 step: single-term outputs 2078
// -> 1491 us per launch, sums 1012 -> 976; FP64 potential at 512x64x128 955 ->
// 831 us, 512x32x32 265 -> 209.  FP64 single-term outputs take
// DFT_XCONV1_COLS64 columns: 16 measured faster than 32, which fill the LDS with
// one block per CU; the accumulating form takes at most 32.)
#ifndef DFT_XCONV1_COLS64
#define DFT_XCONV1_COLS64 16
#endif
template <typename T, int N, bool ONE>
using XConvCfg = ColCfg<T, N, N >= 512 ? 16 : (ONE ? DFT_XCONV1_EM : DFT_XCONV_EM),
                        N >= 512 ? 8
                                 : (ONE ? (sizeof(T) == 8 ? DFT_XCONV1_COLS64 : DFT_XCONV1_COLS)
                                        : (sizeof(T) == 8 && DFT_XCONV_COLS > 32 ? 32 : DFT_XCONV_COLS)),
                        !(ONE && N == 128)>;

template <typename T, int N, bool ONE>
__global__ void __launch_bounds__((XConvCfg<T, N, ONE>::BS), sizeof(T) == 4 ? DFT_XCONV_MINB : DFT_XCONV_MINB64)
    k_xconv(const cplx<T> *__restrict__ g_tw, int nl, int ny, int P, int PP,
            const std::conditional_t<ONE, XOnes, XSum> pg) {
  using C = cplx<T>;
  using G = XConvCfg<T, N, ONE>;
  constexpr int E = G::E, TPL = G::TPL, COLS = G::COLS, LP = G::LP;
  __shared__ C s_x[G::S > 1 ? COLS * LP : 1];
  __shared__ C s_tw[rf::tw_len<T, N>()];
  const int col = threadIdx.x % COLS, t = threadIdx.x / COLS;
  const MidCol mc = mid_col<COLS>(ny, P, nl, col);
  const int o = mc.o, kz = mc.kz;
  const bool act = mc.act;
  const uint32_t es = (uint32_t)ny * PP;
  const uint32_t e0 = (uint32_t)o * PP + kz + t * es;  // element index of point t
  const uint32_t obC = e0 * (uint32_t)sizeof(C), obR = e0 * (uint32_t)sizeof(T);
  const size_t stC = (size_t)TPL * es * sizeof(C), stR = (size_t)TPL * es * sizeof(T);  // per point i
  C *X = s_x + col * LP;
  rf::load_tw<T, N, G::EM, G::BS>(s_tw, g_tw);
  if constexpr (ONE) {
    // single-term outputs: transform, scale and transform back in place
    const auto &tm = pg.o[mc.m];
    C v[E];
    T k[E];
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = rf::gld<C>((const char *)tm.in + i * stC, obC);
#pragma unroll
    for (int i = 0; i < E; ++i) k[i] = rf::gld<T>((const char *)tm.kern + i * stR, obR);
    __syncthreads();
    rf::rfft_apply<T, N, G::EM, rf::BlockSync>(v, X, s_tw, t, [&](int i, double2 u) {
      const double sc = tm.scale * (double)k[i];
      return make_double2(sc * u.x, sc * u.y);
    });
    if (act)
#pragma unroll
      for (int i = 0; i < E; ++i) rf::gst<C>((char *)tm.out + i * stC, obC, v[i]);
  } else {
    C acc[E];
#pragma unroll
    for (int i = 0; i < E; ++i) acc[i] = cmk<C>(0, 0);
    // term q's input and kernel; with DFT_XCONV_PF (FP32) term q + 1's are read
    // before term q's transform
    constexpr bool PF = sizeof(T) == 4 && DFT_XCONV_PF;
    C nv[PF ? E : 1];
    T nk[PF ? E : 1];
    auto fetch = [&](int qq, C *fv, T *fk) {
      const auto &tq = pg.t[qq];
#pragma unroll
      for (int i = 0; i < E; ++i) fv[i] = rf::gld<C>((const char *)tq.in + i * stC, obC);
#pragma unroll
      for (int i = 0; i < E; ++i) fk[i] = rf::gld<T>((const char *)tq.kern + i * stR, obR);
    };
    if constexpr (PF) fetch(0, nv, nk);
    for (int q = 0; q < pg.nterms; ++q) {
      C v[E];
      T k[E];
      if constexpr (PF) {
#pragma unroll
        for (int i = 0; i < E; ++i) v[i] = nv[i], k[i] = nk[i];
        if (q + 1 < pg.nterms) fetch(q + 1, nv, nk);
      } else {
        fetch(q, v, k);
      }
      if (q == 0) __syncthreads();  // twiddles
      rf::rfft<T, N, G::EM, -1, rf::BlockSync>(v, X, s_tw, t);
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const T sc = (T)pg.t[q].scale * k[i];
        acc[i] = cadd(acc[i], cmk<C>(sc * v[i].x, sc * v[i].y));
      }
    }
    rf::rfft<T, N, G::EM, +1, rf::BlockSync>(acc, X, s_tw, t);
    if (act)
#pragma unroll
      for (int i = 0; i < E; ++i) rf::gst<C>((char *)pg.out + i * stC, obC, acc[i]);
  }
}

// ------------------------------------------------------------------- zAB --
// Early loads in zAB, zBC and zC, so that memory round trips overlap the
// transforms: the next stage's spectrum before the current stage's transform,
// the density gradient along the next axis (zAB with KC alone) before the
// current one, the accumulated fields (zBC) before the last transform, the
// step's fields of a line (zC) before the preceding one.
// FP32 only: FP64 holds twice the registers and gains nothing (zBC 433 and 443
// us at 256^3, zAB with KC alone 68.3 and 70.5 at 128x128x256).  The stencils
// are taken after the transforms: loaded before, they cost registers for
// nothing (zAB 297 us at 256^3 FP32 either way, zBC 217 against 213).
template <typename T> constexpr bool early_loads() { return sizeof(T) == 4; }

// Pipelined c2r stages: the spectrum of the current stage was loaded into
// `raw` earlier; the next stage's loads (if any) are issued before this
// stage's transform.
template <typename T, int N>
__device__ __forceinline__ void c2r_pipe(rf::Regs<T, N, pair_em<N>()> &v, fft::RawPair<T, N, pair_em<N>()> &raw,
                                         cplx<T> *X, const cplx<T> *tw, int t, const void *next, uint32_t p, int P) {
  fft::merge_raw<T, N, pair_em<N>()>(v, raw, t);
  if (next) fft::load_raw<T, N, pair_em<N>()>(raw, next, p, P, t);
  rf::rfft<T, N, pair_em<N>(), +1, PairSync<N>>(v, X, tw, t);
}
struct ZABArgs {
  Ptrs8 in;       // rhobar, [rhot], [A, Bx, By, Bz, C] (C null: its term is summed in k space, see fused_impl)
  Ptrs8 out;      // Q, [G_x, G_y, G_z]
  const void *rho, *psi;
  void *rhot, *vre, *vim, *wx, *wy, *wz;
};

// HB: the backflow density switch of HD / HD2 (A, B_d, C come from rho~; Re
// V_BF is multiplied by d(G rho)/d rho, the gradient half of Im V_BF takes rho~).
// Bound by its loads and stores: with KC and backflow 7 spectra and psi in, 4
// spectra and 6 real fields out.  psi of the points is kept, and their density
// and its neighbours' come from psi, so a point takes 4 loads of psi instead of
// 9 of psi and 14 of rho; G_d is formed with the axis' velocity, from the same
// stencil.  With the sums settled after each axis (settle) it takes 160 VGPRs in
// FP32 (231 before) and, at two waves per SIMD, 247 in FP64 (two kernels of 256 +
// 72 and 128 before).  Before and after at 256^3 (us): FP32 388 -> 297, FP64
// 786 -> 516, FP32 with the switch at 256x128x256 261 -> 231.
template <typename T, int N, bool KC, bool BF, bool HB>
__device__ __forceinline__ void zAB_body(ZABArgs a, int64_t npairs, int P, PW<T> pw,
                                         const cplx<T> *__restrict__ g_tw) {
  FUSED_PAIR_SETUP();
  constexpr bool PF = early_loads<T>();
  constexpr int IA = KC ? 2 : 1;  // first backflow input
  const void *rho = a.rho, *psi = a.psi;
  C v[E];
  T vre[2][E];
  fft::RawPair<T, N, pair_em<N>()> raw;
  // c2r of stage input `cur`, then (with early loads) those of `next`
  auto c2r = [&](const void *cur, const void *next) {
    if constexpr (PF) c2r_pipe<T, N>(v, raw, X, s_tw, t, next, p, P);
    else load_c2r<T, N>(v, X, s_tw, t, cur, p, P);
  };
  if constexpr (PF) fft::load_raw<T, N, pair_em<N>()>(raw, a.in.p[BF && KC ? 1 : (BF ? IA : 0)], p, P, t);
  // local correlation: rhobar = Pi*rho, Q; r: the density at the points
  auto local = [&](auto &&dens, const void *next) {
    T r[2][E];
    if constexpr (PF) dens(r);
    c2r(a.in.p[0], next);
    if constexpr (!PF) dens(r);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      T Q[2];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const T rb = part(v[i], w);
        T loc = rb * rb * (pw.c2 * (T)0.5) + rb * rb * rb * (pw.c3 / (T)3);
        if (pw.hdC != (T)0) loc += hd_pot(r[w][i], pw);
        if constexpr (BF) vre[w][i] += loc;
        else vre[w][i] = loc;
        settle(vre[w][i]);
        Q[w] = (rb * pw.c2 + rb * rb * pw.c3) * r[w][i];
      }
      v[i] = cmk<C>(Q[0], Q[1]);
    }
    r2c_store<T, N>(v, X, s_tw, t, a.out.p[0], p, P, act);
  };
  // rhot = F*rho (stored), rho_st = 1 - rhot/rho_0s
  T rst[2][KC ? E : 1];
  auto kc_rst = [&](const void *next) {
    c2r(a.in.p[1], next);
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        rst[w][i] = part(v[i], w) * (-pw.inv_rho0s) + (T)1;
        if (act) q.template put<T>(a.rhot, w, i, part(v[i], w));
      }
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) settle(rst[w][i]);
  };
  // G_d = (D_d rho) rho_st
  auto kc_g = [&](int dd, const T (&g)[2][E]) {
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = cmk<C>(g[0][i] * rst[0][i], g[1][i] * rst[1][i]);
    r2c_store<T, N>(v, X, s_tw, t, a.out.p[1 + dd], p, P, act);
  };
  if constexpr (BF) {
    // A = U*rho; per axis: B_d = U*q_d -> W_d = v_d A - B_d (stored),
    // BF real part sum_d (v_d^2 A - 2 v_d B_d) + C, imaginary part sum_d g_d W_d / (2 (rho+eps)).
    // psi of the points is kept for the three axes; the densities of the
    // neighbours are those of the psi that the velocities load.
    C sp[2][E];
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) sp[w][i] = q.template at<C>(psi, w, i);
    if constexpr (KC) kc_rst(a.in.p[IA]);
    T A[2][E], tr[2][E], im[2][E];
    c2r(a.in.p[IA], a.in.p[IA + 1]);
    // velocity factor per point, kept for the three axes
    T fv[2][E];
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        A[w][i] = part(v[i], w);
        fv[w][i] = velocity_factor(pw, dens_of<T>(sp[w][i]));
        settle(fv[w][i]);
      }
    auto axis = [&](auto dtag) {
      constexpr int D = decltype(dtag)::value;
      void *wd = D == 0 ? a.wx : (D == 1 ? a.wy : a.wz);
      // velocity, density gradient (KC) and gradient of the backflow density
      T vd[2][E], g[2][E], gb[2][HB ? E : 1];
      auto stencil = [&] {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          C na[E], nb[E];
          neighbours<D>(psi, q.here(), sp, w, na, nb);
#pragma unroll
          for (int i = 0; i < E; ++i) {
            vd[w][i] = velocity_sab(pw, fv[w][i], sp[w][i], na[i], nb[i]);
            const T ra = dens_of<T>(na[i]), rb = dens_of<T>(nb[i]);
            g[w][i] = (ra - rb) * pw.inv2h;
            if constexpr (HB) gb[w][i] = (bf_rt(ra, pw) - bf_rt(rb, pw)) * pw.inv2h;
            settle(vd[w][i]), settle(g[w][i]);
            if constexpr (HB) settle(gb[w][i]);
          }
        }
      };
      const void *next = D < 2 || a.in.p[IA + 4] ? a.in.p[D < 2 ? IA + 2 + D : IA + 4] : a.in.p[0];
      c2r(a.in.p[IA + 1 + D], next);
      stencil();
#pragma unroll
      for (int i = 0; i < E; ++i)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const T Bd = part(v[i], w), vw = vd[w][i];
          const T W = vw * A[w][i] - Bd;
          const T ti = vw * vw * A[w][i] + (T)-2 * vw * Bd;
          const T ii = (HB ? gb[w][HB ? i : 0] : g[w][i]) * W;
          tr[w][i] = D == 0 ? ti : tr[w][i] + ti;
          im[w][i] = D == 0 ? ii : im[w][i] + ii;
          settle(tr[w][i]), settle(im[w][i]);
          if (act) q.template put<T>(wd, w, i, W);
        }
      if constexpr (KC) kc_g(D, g);
    };
    axis(std::integral_constant<int, 0>{});
    axis(std::integral_constant<int, 1>{});
    axis(std::integral_constant<int, 2>{});
    const void *C_ = a.in.p[IA + 4];
    if (C_) c2r(C_, a.in.p[0]);
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        T re = tr[w][i];
        if (C_) re += part(v[i], w);
        const T r = dens_of<T>(sp[w][i]);
        if constexpr (HB) re = re * bf_dg(r, pw);
        re = re * ((T)-0.5 * pw.mass);
        if (pw.clamp_bf) re = clampv(re, pw.bfmax);
        vre[w][i] = re * pw.cbf;
        settle(vre[w][i]);
        if (act) q.template put<T>(a.vim, w, i, im[w][i] * ((T)0.5 / (r + pw.div_eps)));
      }
    local([&](T (&r)[2][E]) {
#pragma unroll
      for (int i = 0; i < E; ++i)
#pragma unroll
        for (int w = 0; w < 2; ++w) r[w][i] = dens_of<T>(sp[w][i]);
    }, nullptr);
  } else {
    T rl[2][E];
    local([&](T (&r)[2][E]) {
      const auto ql = q.here();
#pragma unroll
      for (int i = 0; i < E; ++i)
#pragma unroll
        for (int w = 0; w < 2; ++w) rl[w][i] = r[w][i] = ql.template at<T>(rho, w, i);
    }, KC ? a.in.p[1] : nullptr);
    if constexpr (KC) {
      T g[2][E];
      auto grad = [&](auto dtag) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          T na[E], nb[E];
          neighbours<decltype(dtag)::value>(rho, q.here(), rl, w, na, nb);
#pragma unroll
          for (int i = 0; i < E; ++i) g[w][i] = (na[i] - nb[i]) * pw.inv2h;
        }
      };
      if constexpr (PF) grad(std::integral_constant<int, 0>{});
      kc_rst(nullptr);
      auto axis = [&](auto dtag) {
        constexpr int D = decltype(dtag)::value;
        if constexpr (!PF) grad(dtag);
#pragma unroll
        for (int i = 0; i < E; ++i) v[i] = cmk<C>(g[0][i] * rst[0][i], g[1][i] * rst[1][i]);
        if constexpr (PF && D < 2) grad(std::integral_constant<int, D + 1>{});
        r2c_store<T, N>(v, X, s_tw, t, a.out.p[1 + D], p, P, act);
      };
      axis(std::integral_constant<int, 0>{});
      axis(std::integral_constant<int, 1>{});
      axis(std::integral_constant<int, 2>{});
    }
  }
  if (act)
#pragma unroll
    for (int i = 0; i < E; ++i) {
      q.template put<T>(a.vre, 0, i, vre[0][i]);
      q.template put<T>(a.vre, 1, i, vre[1][i]);
    }
}
template <typename T, int N, bool KC, bool BF>
__global__ void __launch_bounds__((PairBS<T, N>), sizeof(T) == 4 ? 0 : 2)
    k_zAB(ZABArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  zAB_body<T, N, KC, BF, false>(a, npairs, P, pw, g_tw);
}
template <typename T, int N, bool KC>
__global__ void __launch_bounds__((PairBS<T, N>), sizeof(T) == 4 ? 0 : 2)
    k_zAB_bfhd(ZABArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  zAB_body<T, N, KC, true, true>(a, npairs, P, pw, g_tw);
}

// ------------------------------------------------------------------- zBC --
struct ZBCArgs {
  Ptrs8 in;   // J_x, J_y, J_z
  Ptrs8 out;  // H
  const void *rho, *rhot, *wx, *wy, *wz;
  void *vre, *vim;
  void *jx, *jy;  // J_x and J_y as real fields, for the rest of sum_d D_d J_d in zC
};

// c2r of the J_d; H = sum_d g_d J_d and its r2c, KC term 3, the z part of term 1
// and the backflow divergence.  KC term 1 is c rst F*(sum_d D_d G_d) = c rst
// sum_d D_d J_d: J_z's difference comes from the line itself (through LDS), J_x
// and J_y are stored for the stencils of zC.  Against a fourth transform for
// the sum, at 256^3 FP32 (us): x-middle 184 -> 116, a y pass of 24 and a z
// transform less, zC 105 -> 133; 32x32x64 FP32 step 91 -> 83.5.
// Bound by the loads: 3 spectra and 7 real fields with stencils (rho and rho~ of
// the points kept for theirs).  With the sums settled after each axis the kernel
// takes 109 VGPRs in FP32 (176 without; 4 waves per SIMD for 2; zBC 268 -> 213
// us at 256^3) and 144 in FP64 (256 and spills, or two kernels with H in memory
// between them, 547 -> 433 us).
// HB: the backflow density switch of HD / HD2 (the divergence half of Im V_BF
// is multiplied by G(rho)).
// GRAD: the energy gradient's form, c sum_d D_d (rst J_d) without term 3: rst J_x
// and rst J_y are stored, the z part added to V_re.
template <typename T, int N, bool BF, bool HB, bool GRAD>
__device__ __forceinline__ void zBC_body(ZBCArgs a, int64_t npairs, int P, PW<T> pw,
                                         const cplx<T> *__restrict__ g_tw) {
  FUSED_PAIR_SETUP();
  constexpr bool PF = early_loads<T>();
  const void *rho = a.rho, *rhot = a.rhot;
  C v[E];
  T H[2][E], t3[2][E];
  fft::RawPair<T, N, pair_em<N>()> raw;
  auto c2r = [&](const void *cur, const void *next) {
    if constexpr (PF) c2r_pipe<T, N>(v, raw, X, s_tw, t, next, p, P);
    else load_c2r<T, N>(v, X, s_tw, t, cur, p, P);
  };
  if constexpr (PF) fft::load_raw<T, N, pair_em<N>()>(raw, a.in.p[0], p, P, t);
  // rho and rho~ of the points, kept for the stencils of the three axes
  T sr[2][E], st[2][E];
#pragma unroll
  for (int i = 0; i < E; ++i)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      sr[w][i] = q.template at<T>(rho, w, i);
      st[w][i] = q.template at<T>(rhot, w, i);
    }
  auto rst = [&](int w, int i) { return st[w][i] * (-pw.inv_rho0s) + (T)1; };
  auto axis = [&](auto dtag) {
    constexpr int D = decltype(dtag)::value;
    T g[E];
    auto diff_w = [&](const void *f, const T (&s)[2][E], int w, T (&out)[E]) {
      T na[E], nb[E];
      neighbours<D>(f, q.here(), s, w, na, nb);
#pragma unroll
      for (int i = 0; i < E; ++i) out[i] = (na[i] - nb[i]) * pw.inv2h;
    };
    c2r(a.in.p[D], D < 2 ? a.in.p[D + 1] : nullptr);
    if constexpr (D < 2)
      if (act)
#pragma unroll
        for (int i = 0; i < E; ++i)
#pragma unroll
          for (int w = 0; w < 2; ++w)
            q.template put<T>(D == 0 ? a.jx : a.jy, w, i, GRAD ? rst(w, i) * part(v[i], w) : part(v[i], w));
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      diff_w(rho, sr, w, g);
#pragma unroll
      for (int i = 0; i < E; ++i) H[w][i] = D == 0 ? g[i] * part(v[i], w) : H[w][i] + g[i] * part(v[i], w);
      if constexpr (!GRAD) {
        diff_w(rhot, st, w, g);  // (dF_d * rho) = D_d (F * rho)
#pragma unroll
        for (int i = 0; i < E; ++i) t3[w][i] = D == 0 ? g[i] * part(v[i], w) : t3[w][i] + g[i] * part(v[i], w);
      }
    }
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int i = 0; i < E; ++i) {
        settle(H[w][i]);
        if constexpr (!GRAD) settle(t3[w][i]);
      }
  };
  // the backflow divergence and V_re so far, with early loads before J_z's transform
  auto bf_div = [&] {
    if constexpr (BF)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const auto qt = q.here();
#pragma unroll
        for (int i = 0; i < E; ++i) {
          T im = qt.template at_once<T>(a.vim, w, i);
          T gw = (T)1;
          if constexpr (HB) gw = bf_g(sr[w][i], pw);
          im += (T)0.5 * (((qt.template nb<T, 0, 1>(a.wx, w, i) - qt.template nb<T, 0, -1>(a.wx, w, i)) * pw.inv2h) * gw);
          im += (T)0.5 * (((qt.template nb<T, 1, 1>(a.wy, w, i) - qt.template nb<T, 1, -1>(a.wy, w, i)) * pw.inv2h) * gw);
          im += (T)0.5 * (((qt.template nb<T, 2, 1>(a.wz, w, i) - qt.template nb<T, 2, -1>(a.wz, w, i)) * pw.inv2h) * gw);
          if (pw.clamp_bf) im = clampv(im, pw.bfmax);
          if (act) qt.template put<T>(a.vim, w, i, im * pw.cbf);
        }
      }
  };
  T base[2][E];
  auto base_w = [&](int w) {
    const auto qt = q.here();
#pragma unroll
    for (int i = 0; i < E; ++i) base[w][i] = qt.template at_once<T>(a.vre, w, i);
  };
  axis(std::integral_constant<int, 0>{});
  axis(std::integral_constant<int, 1>{});
  if constexpr (PF) bf_div(), base_w(0), base_w(1);
  axis(std::integral_constant<int, 2>{});
  // D_z J_z (GRAD: of rst J_z) from the neighbouring points of both lines
  using LY = rf::LayOf<T, N, pair_em<N>(), PairSync<N>>;
  C dz[E];
#pragma unroll
  for (int i = 0; i < E; ++i) X[LY::pad(t + TPL * i)] = GRAD ? cmk<C>(rst(0, i) * v[i].x, rst(1, i) * v[i].y) : v[i];
  PairSync<N>::sync();
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int z = t + TPL * i;
    dz[i] = cscale(csub(X[LY::pad((z + 1) & (N - 1))], X[LY::pad((z - 1) & (N - 1))]), pw.inv2h);
  }
  PairSync<N>::sync();
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    if constexpr (!PF) base_w(w);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      T kc;
      if constexpr (GRAD) kc = part(dz[i], w) * pw.ckc;
      else kc = part(dz[i], w) * rst(w, i) * pw.ckc - t3[w][i] * (pw.ckc * pw.k23);
      if (act) q.template put<T>(a.vre, w, i, base[w][i] + kc);
    }
  }
#pragma unroll
  for (int i = 0; i < E; ++i) v[i] = cmk<C>(H[0][i], H[1][i]);
  r2c_store<T, N>(v, X, s_tw, t, a.out.p[0], p, P, act);
  if constexpr (!PF) bf_div();
}
template <typename T, int N, bool BF>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zBC(ZBCArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  zBC_body<T, N, BF, false, false>(a, npairs, P, pw, g_tw);
}
template <typename T, int N>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zBC_bfhd(ZBCArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  zBC_body<T, N, true, true, false>(a, npairs, P, pw, g_tw);
}

template <typename T, int N>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zBC_grad(ZBCArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  zBC_body<T, N, false, false, true>(a, npairs, P, pw, g_tw);
}

// Last stage of the energy gradient: c2r of the linear terms, V_re and (KC) the
// differences of M_x = rst J_x and M_y added.
template <typename T, int N, bool KC>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zG(const void *lin, const void *vre, const void *mx, const void *my, T *grad, int64_t npairs, int P, PW<T> pw,
         const cplx<T> *__restrict__ g_tw) {
  FUSED_PAIR_SETUP();
  C v[E];
  load_c2r<T, N>(v, X, s_tw, t, lin, p, P);
  const auto qq = q.here();
#pragma unroll
  for (int w = 0; w < 2; ++w)
#pragma unroll
    for (int i = 0; i < E; ++i) {
      T g = qq.template at_once<T>(vre, w, i) + part(v[i], w);
      if constexpr (KC)
        g += ((qq.template nb<T, 0, 1>(mx, w, i) - qq.template nb<T, 0, -1>(mx, w, i)) +
              (qq.template nb<T, 1, 1>(my, w, i) - qq.template nb<T, 1, -1>(my, w, i))) *
             pw.inv2h * pw.ckc;
      if (act) q.template put<T>(grad, w, i, g);
    }
}

// -------------------------------------------------------------------- zC --
// Kernel arguments are fetched when a wavefront starts, and on small grids that is
// part of a launch's time: kept to what the kernel reads, most used first (plain
// step at 64^3 FP64: zC 9.5 us with the whole PW, 384 bytes of arguments, 8.6 with
// these 184).
struct ZCArgs {
  const void *in;         // summed linear terms (half spectrum)
  const void *vre, *vim;  // vim null without backflow
  // step mode
  const void *vext;      // real, may be null
  double mu;
  const void *vavg;      // complex, may be null: V_eff = (vavg + V_eff)/2
  void *vsave;           // complex, may be null: stores V_eff before averaging
  void *phase;           // complex out: V_eff of the step (the inverse z pass applies e^{-i V_eff dt/2})
  const void *psi_src;
  void *psi_dst;         // z forward transform of psi_src * phase
  double dtr, dti;
  void *V;               // API mode: potential accumulated here
  const void *jx, *jy, *rhot;  // KC: J_x, J_y (the x and y parts of term 1) and F*rho
  int nx, ny;                  // and the values of PW that it takes
  double inv2h, inv_rho0s, ckc;
};

template <typename T, int N, bool STEP, bool KC>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zC(const cplx<T> *__restrict__ g_tw, int64_t npairs, int P, ZCArgs a) {
  using C = cplx<T>;
  using G = LineCfg<T, N, pair_em<N>()>;
  constexpr int E = G::E, TPL = G::TPL, LP = G::LP;
  __shared__ C s_x[G::LINES * LP];
  __shared__ C s_tw[rf::tw_len<T, N>()];
  const int ln = threadIdx.x / TPL, t = threadIdx.x % TPL;
  const uint32_t p0 = (uint32_t)blockIdx.x * G::LINES + ln;
  const bool act = p0 < npairs;
  const uint32_t p = act ? p0 : 0;
  C *X = s_x + ln * LP;
  rf::load_tw<T, N, G::EM, G::BS>(s_tw, g_tw);
  __syncthreads();
  constexpr bool PF = early_loads<T>();
  C v[E];
  auto c2r_in = [&] { load_c2r<T, N>(v, X, s_tw, t, a.in, p, P); };
  const uint32_t cb = p * 2u * N + (uint32_t)t;
  const PairPos<T, N, TPL> q(p, t, a.nx, a.ny);
  // the x and y parts of KC term 1, c rst (D_x J_x + D_y J_y), in two parts: the
  // loads of line w, and its value at point i
  T jd[KC ? 4 : 1][KC ? E : 1], rt[KC ? E : 1];
  auto t1_fetch = [&](int w) {
    if constexpr (KC) {
      const auto qq = q.here();
#pragma unroll
      for (int i = 0; i < E; ++i) {
        jd[0][i] = qq.template nb<T, 0, 1>(a.jx, w, i);
        jd[1][i] = qq.template nb<T, 0, -1>(a.jx, w, i);
        jd[2][i] = qq.template nb<T, 1, 1>(a.jy, w, i);
        jd[3][i] = qq.template nb<T, 1, -1>(a.jy, w, i);
        rt[i] = qq.template at_once<T>(a.rhot, w, i);
      }
    }
  };
  auto t1 = [&](int i) {
    if constexpr (KC)
      return ((jd[0][i] - jd[1][i]) + (jd[2][i] - jd[3][i])) * (T)a.inv2h * (rt[i] * (T)-a.inv_rho0s + (T)1) * (T)a.ckc;
    else return (T)0;
  };
  if constexpr (!STEP) {
    c2r_in();
    const uint32_t c0 = cb + rf::opaque_zero();
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      t1_fetch(w);
      if (act)
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const int d = w * N + TPL * i;
          C u = rf::lde<C>(a.V, c0, d);
          u.x += (rf::lde<T>(a.vre, c0, d) + t1(i)) + part(v[i], w);
          u.y += a.vim ? rf::lde<T>(a.vim, c0, d) : (T)0;
          rf::ste<C>(a.V, c0, u, d);
        }
    }
  } else {
    // the fields of line w; with prefetching, line 0's are read before the
    // transform above and line 1's before line 0's transform
    T bre[E], bim[E], bex[E];
    C bav[E], bps[E];
    auto fetch = [&](int w) {
      t1_fetch(w);
      const uint32_t c0 = cb + rf::opaque_zero();
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int d = w * N + TPL * i;
        bre[i] = rf::lde_once<T>(a.vre, c0, d);
        bim[i] = a.vim ? rf::lde_once<T>(a.vim, c0, d) : (T)0;
        bex[i] = a.vext ? rf::lde_once<T>(a.vext, c0, d) : (T)0;
        if (a.vavg) bav[i] = rf::lde_once<C>(a.vavg, c0, d);
        bps[i] = rf::lde_once<C>(a.psi_src, c0, d);
      }
    };
    if constexpr (PF) fetch(0);
    c2r_in();
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      if constexpr (!PF) fetch(w);
      const uint32_t c0 = cb + rf::opaque_zero();
      C u[E], ph[E], vs[E];  // ph: the potential of this half step (re-applied by the inverse z pass)
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const T re = (bre[i] + t1(i)) + part(v[i], w);
        const T im = bim[i];
        C ve = cmk<C>(re - (T)a.mu + bex[i], im);
        if (a.vsave) vs[i] = ve;
        if (a.vavg) {
          const C va = bav[i];
          ve = cmk<C>((va.x + ve.x) * (T)0.5, (va.y + ve.y) * (T)0.5);
        }
        ph[i] = ve;
        u[i] = fft::apply_vphase<T>(bps[i], ve, a.dtr, a.dti);
      }
      if (act) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          rf::ste<C>(a.phase, c0, ph[i], w * N + TPL * i);
          if (a.vsave) rf::ste<C>(a.vsave, c0, vs[i], w * N + TPL * i);
        }
      }
      if constexpr (PF) {
        if (w == 0) fetch(1);
      }
      rf::rfft<T, N, pair_em<N>(), -1, PairSync<N>>(u, X, s_tw, t);
      if (act)
#pragma unroll
        for (int i = 0; i < E; ++i) rf::ste<C>(a.psi_dst, c0, u[i], w * N + TPL * i);
    }
  }
}

// -------------------------------------------------------------------- zE --
struct ZEArgs {
  Ptrs8 in;   // LJ*rho, rhobar, [rhot], [A, B_x, B_y, B_z, C]; k_zE2: J_x, J_y, J_z
  Ptrs8 out;  // [G_x, G_y, G_z]
  const void *rho, *psi;
  void *rhot, *eps;
};

// The energy density without its KC part, from the convolutions of zA's fields:
// local terms, backflow -m c_bf/4 (A v^2 + C) rho + m c_bf/2 sum_d B_d rho v_d
// (rho~ = G rho in place of rho with the switch, HB), and the r2c of G_d =
// (D_d rho) rho_st.  In this way no convolution, velocity or gradient goes
// through memory as a real field.  psi (with KC alone: rho) of the points is
// kept for the stencils, as in zAB; bound by the loads of the spectra.
template <typename T, int N, bool KC, bool BF, bool HB>
__device__ __forceinline__ void zE_body(ZEArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  FUSED_PAIR_SETUP();
  constexpr bool PF = early_loads<T>();
  constexpr int IA = KC ? 3 : 2;  // first backflow input
  C v[E];
  fft::RawPair<T, N, pair_em<N>()> raw;
  auto c2r = [&](const void *cur, const void *next) {
    if constexpr (PF) c2r_pipe<T, N>(v, raw, X, s_tw, t, next, p, P);
    else load_c2r<T, N>(v, X, s_tw, t, cur, p, P);
  };
  if constexpr (PF) fft::load_raw<T, N, pair_em<N>()>(raw, a.in.p[KC ? 2 : (BF ? IA + 1 : 0)], p, P, t);
  // psi of the points (backflow), or their density
  using S = std::conditional_t<BF, C, T>;
  const void *src = BF ? a.psi : a.rho;
  S sp[2][E];
  T e[2][E], rst[2][KC ? E : 1];
#pragma unroll
  for (int i = 0; i < E; ++i)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      sp[w][i] = q.template at<S>(src, w, i);
      e[w][i] = 0;
    }
  auto dens = [&](const S &s) {
    if constexpr (BF) return dens_of<T>(s);
    else return s;
  };
  if constexpr (KC) {
    c2r(a.in.p[2], BF ? a.in.p[IA + 1] : a.in.p[0]);
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        rst[w][i] = part(v[i], w) * (-pw.inv_rho0s) + (T)1;
        settle(rst[w][i]);
        if (act) q.template put<T>(a.rhot, w, i, part(v[i], w));
      }
  }
  const T mq = pw.cbf * pw.mass * (T)0.25, mh = pw.cbf * pw.mass * (T)0.5;
  T fv[2][BF ? E : 1], rw[2][BF ? E : 1], v2[2][BF ? E : 1];
  if constexpr (BF)
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const T r = dens(sp[w][i]);
        fv[w][i] = velocity_factor(pw, r);
        rw[w][i] = HB ? bf_rt(r, pw) : r;
        v2[w][i] = 0;
        settle(fv[w][i]), settle(rw[w][i]);
      }
  auto axis = [&](auto dtag) {
    constexpr int D = decltype(dtag)::value;
    if constexpr (BF) c2r(a.in.p[IA + 1 + D], a.in.p[D < 2 ? IA + 2 + D : IA]);
    T g[2][E];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      S na[E], nb[E];
      neighbours<D>(src, q.here(), sp, w, na, nb);
#pragma unroll
      for (int i = 0; i < E; ++i) {
        if constexpr (BF) {
          const T vd = velocity_sab(pw, fv[w][i], sp[w][i], na[i], nb[i]);
          v2[w][i] += vd * vd;
          e[w][i] += mh * (part(v[i], w) * rw[w][i] * vd);
          settle(v2[w][i]), settle(e[w][i]);
        }
        if constexpr (KC) g[w][i] = (dens(na[i]) - dens(nb[i])) * pw.inv2h * rst[w][i];
      }
    }
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = cmk<C>(g[0][i], g[1][i]);
      r2c_store<T, N>(v, X, s_tw, t, a.out.p[D], p, P, act);
    }
  };
  if constexpr (KC || BF) {
    axis(std::integral_constant<int, 0>{});
    axis(std::integral_constant<int, 1>{});
    axis(std::integral_constant<int, 2>{});
  }
  // the remaining convolutions, each weighted with a field at the points
  auto add = [&](const void *cur, const void *next, auto &&f) {
    c2r(cur, next);
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        e[w][i] += f(w, i, part(v[i], w));
        settle(e[w][i]);
      }
  };
  if constexpr (BF) {
    add(a.in.p[IA], a.in.p[IA + 4], [&](int w, int i, T A) { return -mq * (A * v2[w][i] * rw[w][i]); });
    add(a.in.p[IA + 4], a.in.p[0], [&](int w, int i, T c) { return -mq * (c * rw[w][i]); });
  }
  add(a.in.p[0], a.in.p[1], [&](int w, int i, T lj) { return (T)0.5 * dens(sp[w][i]) * lj; });
  add(a.in.p[1], nullptr, [&](int w, int i, T rb) {
    const T r = dens(sp[w][i]);
    T loc = (pw.c2 * (T)0.5) * (rb * rb * r) + (pw.c3 / (T)3) * (rb * rb * rb * r);
    if (pw.hdC != (T)0) loc += hd_eps(r, pw);
    return loc;
  });
  if (act)
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) q.template put<T>(a.eps, w, i, e[w][i]);
}
template <typename T, int N, bool KC, bool BF, bool HB>
__global__ void __launch_bounds__((PairBS<T, N>), sizeof(T) == 4 ? 0 : 2)
    k_zE(ZEArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  zE_body<T, N, KC, BF, HB>(a, npairs, P, pw, g_tw);
}

// KC part of the energy density: eps -= (alpha_s / 4m) rho_st sum_d (D_d rho) J_d
template <typename T, int N>
__global__ void __launch_bounds__((PairBS<T, N>), 0)
    k_zE2(ZEArgs a, int64_t npairs, int P, PW<T> pw, const cplx<T> *__restrict__ g_tw) {
  FUSED_PAIR_SETUP();
  constexpr bool PF = early_loads<T>();
  C v[E];
  T sr[2][E], H[2][E];
  fft::RawPair<T, N, pair_em<N>()> raw;
  if constexpr (PF) fft::load_raw<T, N, pair_em<N>()>(raw, a.in.p[0], p, P, t);
#pragma unroll
  for (int i = 0; i < E; ++i)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      sr[w][i] = q.template at<T>(a.rho, w, i);
      H[w][i] = 0;
    }
  auto axis = [&](auto dtag) {
    constexpr int D = decltype(dtag)::value;
    if constexpr (PF) c2r_pipe<T, N>(v, raw, X, s_tw, t, D < 2 ? a.in.p[D + 1] : nullptr, p, P);
    else load_c2r<T, N>(v, X, s_tw, t, a.in.p[D], p, P);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      T na[E], nb[E];
      neighbours<D>(a.rho, q.here(), sr, w, na, nb);
#pragma unroll
      for (int i = 0; i < E; ++i) {
        H[w][i] += (na[i] - nb[i]) * pw.inv2h * part(v[i], w);
        settle(H[w][i]);
      }
    }
  };
  axis(std::integral_constant<int, 0>{});
  axis(std::integral_constant<int, 1>{});
  axis(std::integral_constant<int, 2>{});
  const auto qt = q.here();
#pragma unroll
  for (int i = 0; i < E; ++i)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const T rst = qt.template at_once<T>(a.rhot, w, i) * (-pw.inv_rho0s) + (T)1;
      const T e = qt.template at_once<T>(a.eps, w, i) - (T)0.5 * pw.ckc * (rst * H[w][i]);
      if (act) qt.template put<T>(a.eps, w, i, e);
    }
}

}  // namespace fused
}  // namespace dft
