// Circulant-embedded BTTB operator on gfx950: kernel-spectrum precompute
// (FP64) and the three fused FFT passes of the matvec.
//
// Reference counterparts: Ghat = FFT(G_prep) at B/CUDA_GMRES/launch_GMRES.cuh:138-142;
// G_x_fft_matvec at B/CUDA_GMRES/Fast_matvec.cuh:1-56, i.e. the chain
// extend_by_zeros_kernel -> cufftExecC2C -> MatMul_ElemWise_kernel ->
// cufftExecC2C -> _2D_to_1D_kernel (B/CUDA_GMRES/GMRES_kernels.cuh:98-167,286-326).
//
// Here the embedding is M x M with M >= 2N-1 chosen FFT-friendly (2^a or
// 3*2^a), and the five reference launches collapse into three passes:
//   pass 1  row i < N:  u = chi .* (s x)[i, :] zero-padded to M, forward FFT
//                       along the row -> T[i, :]      (optionally writes s x back)
//   pass 2  column c:   forward FFT of T[:, c] (rows >= N are zero), multiply
//                       by Ghat[:, c], inverse FFT, keep rows < N -> T[:, c]
//   pass 3  row i < N:  inverse FFT of T[i, :], crop to N, scale 1/M^2 and
//                       combine with x (and b for a residual) -> y[i, :]
// T is N x M in column panels (tpos), so only N of the M rows are ever stored.
//
// The passes hold their transforms in registers and cross threads through LDS
// between stages only (cgm_fft.h): S stages take S - 1 exchanges, where transforms
// kept in LDS took S + 1.  N = 301, two vectors: 33.4 -> 23.0 us; N = 512, one
// vector: 25 -> 20.6 us (replays of a graph; 5.0 + 7.9 + 5.2 in the passes alone),
// 16 vectors: 124 -> 105 us (20 + 50 + 26; pass 2 is bound by its vector arithmetic, 35
// us at full issue, passes 1 and 3 by memory).
#include <math.h>
#include <string.h>

#include "cgm_fft.h"
#include "cgm_internal.h"
#include "cgm_special.h"

namespace cgm {

// ---------------------------------------------------------------------------
// pass kernels
// ---------------------------------------------------------------------------
// Work-group bound: float kernels accept tiles up to 1024 threads (autotuned
// rows/columns per work-group); double kernels keep the tighter bound that
// avoids register spills of the FP64 transforms.
// Elements per thread of the pass kernels: 16 saves one of four stages at 2048
// and 4096 points in single precision (N = 1024, four vectors: 133.6 against 149.1
// us); at 128-512 points the fewer waves cost more (N = 128, one vector: 13.3
// against 10.0 us), and so do the registers of 16 double elements (N = 1024:
// 88.8 against 83.2 us) and of 24 elements at 3 * 2^k (N = 384, four vectors: 48.0
// against 40.0 us).
template <typename T, int M> constexpr int kPassE = sizeof(T) == 4 && (M == 2048 || M == 4096) ? 16 : kFftE<M>;
// At M = 1024 in single precision both 8 and 16 pay, by pass and batch (the
// autotuner's radix plan): with 16 a transform is one wave (radices 16, 8, 8),
// with 8 two waves and a stage more.
constexpr int kWideE = 16;
template <typename T, int M, int E> struct PassWG {
  using Shape = FftShape<M, E>;
  static constexpr int want = sizeof(T) == 8 ? 0 : E == 8 ? 1024 : 0;
  static constexpr int value = Shape::WG > want ? Shape::WG : want;
};

template <typename T, int M, int E>
__global__ void __launch_bounds__((PassWG<T, M, E>::value))
k_pass1(const cplx<T>* __restrict__ x, cplx<T>* xw, const T* __restrict__ chi,
        const double* __restrict__ norm_ptr, int mode, cplx<T>* __restrict__ Tm, int N,
        int rows_per_wg, const cplx<T>* __restrict__ tw, const int* __restrict__ done, BatchStrides bs) {
  {
    const long k = blockIdx.y;
    x += k * bs.x;
    if (xw) xw += k * bs.x;
    if (chi) chi += k * bs.chi;
    Tm += k * bs.T;
    norm_ptr = boff(norm_ptr, k * bs.st);
    done = boff(done, k * bs.st);
  }
  const int dn = done ? *done : 0;  // tested once the row loads are in flight
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* smem = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int NT = FftShape<M, E>::NT;
  constexpr int EPT = E;
  const int t = threadIdx.x % NT;
  const int rl = threadIdx.x / NT;
  const int row = blockIdx.x * rows_per_wg + rl;
  cplx<T>* buf = smem + rl * LdsLen<M>::value;
  const bool live = row < N;
  const long rb = (long)row * N;
  const bool mul = mode == kModeForward || mode == kModeResidual;
  FftTwiddles<T, M, E> tws;
  tws.load(tw, t);
  // the row is zero from N <= M/2 on: registers EPT/2 .. stay unused
  cplx<T> v[EPT];
  T cv[EPT / 2];
#pragma unroll
  for (int k = 0; k < EPT / 2; ++k) {
    const int e = t + k * NT;
    v[k] = (live && e < N) ? x[rb + e] : mk(T(0), T(0));
    cv[k] = (live && e < N && mul) ? chi[rb + e] : T(1);
  }
  if (dn) return;
  T s = T(1);
  if (norm_ptr) {
    const double nv = *norm_ptr;
    s = nv > 0.0 ? T(1.0 / nv) : T(0);
  }
#pragma unroll
  for (int k = 0; k < EPT / 2; ++k) {
    const int e = t + k * NT;
    if (norm_ptr) {
      v[k] = cscale(v[k], s);
      if (xw && live && e < N) xw[rb + e] = v[k];
    }
    if (mul) v[k] = cscale(v[k], cv[k]);
  }
  reg_fft<T, M, -1, true, false, E>(v, buf, tws, t);
  if (live) {
#pragma unroll
    for (int k = 0; k < EPT; ++k) Tm[tpos(row, t + k * NT, N)] = v[k];
  }
}

template <typename T, typename G, int M, int E>
__global__ void __launch_bounds__((PassWG<T, M, E>::value))
k_pass2(cplx<T>* __restrict__ Tm, const G* __restrict__ gq, int N, int cols_per_wg,
        const cplx<T>* __restrict__ tw, const int* __restrict__ done, BatchStrides bs) {
  Tm += (long)blockIdx.y * bs.T;
  done = boff(done, (long)blockIdx.y * bs.st);
  const int dn = done ? *done : 0;  // tested once the column loads are in flight
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* smem = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int NT = FftShape<M, E>::NT;
  constexpr int EPT = E;
  constexpr int H = M / 2 + 1;
  constexpr int ML = LdsLen<M>::value;
  const int grp = xcd_tile(blockIdx.x, gridDim.x);
  const int c0 = grp * cols_per_wg;
  const int t = threadIdx.x % NT;
  const int cl = threadIdx.x / NT;
  FftTwiddles<T, M, E> tws;
  tws.load(tw, t);
  // gather the column tile: consecutive threads read consecutive columns; N <=
  // M/2, so each thread gathers at most EPT/2 values, of column c and rows r0 + k NT
  // (the work-group is cols_per_wg * NT threads).  A division by cols_per_wg for
  // each value was a third of the kernel's vector instructions (M = 1024, one wave
  // per column: 2,007 of them, now 1,320).
  constexpr int GR = EPT / 2;
  const int r0 = threadIdx.x / cols_per_wg, c = threadIdx.x - r0 * cols_per_wg;
  {
    cplx<T> gv[GR];
#pragma unroll
    for (int k = 0; k < GR; ++k) {
      const int r = r0 + k * NT;
      if (r < N) gv[k] = Tm[tpos(r, c0 + c, N)];
    }
    if (dn) return;
#pragma unroll
    for (int k = 0; k < GR; ++k) {
      const int r = r0 + k * NT;
      if (r < N) smem[c * ML + lpad(r)] = gv[k];
    }
  }
  // the column's multipliers, loaded ahead of the transform
  const int col = c0 + cl;
  const int cq = col <= M - col ? col : M - col;
  const G* grow = gq + (long)cq * H;
  G g[EPT];
  const auto load_g = [&] {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int e = t + k * NT;
      g[k] = grow[e <= M - e ? e : M - e];
    }
  };
  if constexpr (!FftTwiddles<T, M, E>::late) load_g();  // else the registers are worth more than the latency
  __syncthreads();
  cplx<T>* buf = smem + cl * ML;
  cplx<T> v[EPT];
#pragma unroll
  for (int k = 0; k < EPT / 2; ++k) {
    const int e = t + k * NT;
    v[k] = e < N ? buf[lpad(e)] : mk(T(0), T(0));
  }
  FftSync<M, E>::stage();
  reg_fft<T, M, -1, true, false, E>(v, buf, tws, t);  // rows N.. are zero
  if constexpr (FftTwiddles<T, M, E>::late) load_g();
  tws.refresh();
#pragma unroll
  for (int k = 0; k < EPT; ++k) v[k] = cmul(v[k], mk(T(g[k].x), T(g[k].y)));
  FftSync<M, E>::stage();
  reg_fft<T, M, +1, false, true, E>(v, buf, tws, t);  // rows < N are kept
  FftSync<M, E>::stage();
#pragma unroll
  for (int k = 0; k < EPT / 2; ++k) {
    const int e = t + k * NT;
    if (e < N) buf[lpad(e)] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < GR; ++k) {
    const int r = r0 + k * NT;
    if (r < N) Tm[tpos(r, c0 + c, N)] = smem[c * ML + lpad(r)];
  }
}

template <typename T, int M, int E>
__global__ void __launch_bounds__((PassWG<T, M, E>::value))
k_pass3(const cplx<T>* __restrict__ Tm, const cplx<T>* __restrict__ x, const T* __restrict__ chi,
        const cplx<T>* __restrict__ b, cplx<T>* __restrict__ y, int mode, int N, int rows_per_wg,
        T inv, const cplx<T>* __restrict__ tw, const int* __restrict__ done, BatchStrides bs) {
  {
    const long k = blockIdx.y;
    Tm += k * bs.T;
    x += k * bs.x;
    if (chi) chi += k * bs.chi;
    if (b) b += k * bs.b;
    y += k * bs.y;
    done = boff(done, k * bs.st);
  }
  const int dn = done ? *done : 0;  // tested once the row loads are in flight
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* smem = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int NT = FftShape<M, E>::NT;
  constexpr int EPT = E;
  const int t = threadIdx.x % NT;
  const int rl = threadIdx.x / NT;
  const int row = blockIdx.x * rows_per_wg + rl;
  cplx<T>* buf = smem + rl * LdsLen<M>::value;
  const bool live = row < N;
  FftTwiddles<T, M, E> tws;
  tws.load(tw, t);
  cplx<T> v[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) v[k] = live ? Tm[tpos(row, t + k * NT, N)] : mk(T(0), T(0));
  if (dn) return;
  reg_fft<T, M, +1, false, true, E>(v, buf, tws, t);  // columns < N are used
  if (!live) return;
  const long rb = (long)row * N;
#pragma unroll
  for (int k = 0; k < EPT / 2; ++k) {
    const int e = t + k * NT;
    if (e >= N) continue;
    const cplx<T> g = cscale(v[k], inv);
    cplx<T> o;
    switch (mode) {
      case kModeForward: o = csub(x[rb + e], g); break;
      case kModeAdjoint: o = csub(x[rb + e], cscale(g, chi[rb + e])); break;
      case kModeGreen: o = g; break;
      case kModeResidual: o = csub(b[rb + e], csub(x[rb + e], g)); break;
      default: o = csub(b[rb + e], csub(x[rb + e], cscale(g, chi[rb + e]))); break;
    }
    y[rb + e] = o;
  }
}

// ---------------------------------------------------------------------------
// The whole product in one launch, for grids whose M x M embedding fits the
// LDS of one work-group with room to spare (complex64: M <= 96, i.e. N <= 48;
// complex128: M <= 64).
// Work-group blockIdx.x takes vector blockIdx.x through the three passes with T
// in LDS: element (r, c) at r * RS + r / 8 + c + c / 8, whose pads keep the
// stage-0 writes (stride 8) of rows and columns off each other's banks.  Every
// transform lies in one wave (FftSync), so the work-group meets only between the
// passes.  The transforms are those of k_pass1..3: results are equal bit for bit.
//
// Such a product is a chain of latencies: three launches that each wait for the
// one before, with a few work-groups each.  N = 24, one vector: 6.6 us instead of
// 10.9 (FP64: 7.4 instead of 13.2).  At N = 48 the two are level: 12.3 us against
// 11.6 in replays of a graph, 12.4 against 13.3 where the host issues the launches.
// At M = 128 one CU's LDS traffic costs more than the launches (N = 64, one
// vector: 15.6 against 9.7 us).
// ---------------------------------------------------------------------------
template <int M> struct SmallShape {
  static constexpr int E = kFftE<M>;
  static constexpr int NT = FftShape<M, E>::NT;
  static constexpr int want = M * NT < 64 ? 64 : (M * NT + 63) / 64 * 64;
  static constexpr int BS = want > 1024 ? 1024 : want;
  static constexpr int RS = M + M / 8 + 1;
  static constexpr int len = M * RS + M / 8;  // elements of T
};
struct LdsGridRow {
  __device__ inline int operator()(int e) const { return e + (e >> 3); }
};
template <int RS> struct LdsGridCol {
  __device__ inline int operator()(int e) const { return e * RS + (e >> 3); }
};

template <typename T, typename G, int M>
__global__ void __launch_bounds__(SmallShape<M>::BS)
k_matvec_small(const cplx<T>* __restrict__ x, const T* __restrict__ chi, const G* __restrict__ gq,
               cplx<T>* __restrict__ y, int mode, int N, T inv, const cplx<T>* __restrict__ tw, BatchStrides bs) {
  using S = SmallShape<M>;
  constexpr int E = S::E, NT = S::NT, EPT = E, PER = S::BS / NT, RS = S::RS, H = M / 2 + 1;
  __shared__ __align__(16) cplx<T> buf[S::len];
  static_assert(FftSync<M, E>::one_wave, "one wave per transform");
  x += (long)blockIdx.x * bs.x;
  if (chi) chi += (long)blockIdx.x * bs.chi;
  y += (long)blockIdx.x * bs.y;
  const int t = threadIdx.x % NT, l = threadIdx.x / NT;
  const bool mul = mode == kModeForward;
  FftTwiddles<T, M, E> tws;
  tws.load(tw, t);
  // rows i < N: chi .* x, forward
  for (int r0 = 0; r0 < N; r0 += PER) {
    const int r = r0 + l;
    const bool live = r < N;
    cplx<T>* row = buf + r * RS + (r >> 3);
    cplx<T> v[EPT];
#pragma unroll
    for (int k = 0; k < EPT / 2; ++k) {
      const int e = t + k * NT;
      const bool in = live && e < N;
      v[k] = in ? x[(long)r * N + e] : mk(T(0), T(0));
      if (mul && in) v[k] = cscale(v[k], chi[(long)r * N + e]);
    }
    reg_fft<T, M, -1, true, false, E>(v, row, tws, t, live, LdsGridRow());
    FftSync<M, E>::stage();
    if (live) {
#pragma unroll
      for (int k = 0; k < EPT; ++k) row[LdsGridRow()(t + k * NT)] = v[k];
    }
  }
  __syncthreads();
  // columns: forward, times the spectrum, inverse
  for (int c0 = 0; c0 < M; c0 += PER) {
    const int c = c0 + l;
    const bool live = c < M;
    cplx<T>* col = buf + c + (c >> 3);
    const int cq = c <= M - c ? c : M - c;
    G g[EPT];
    cplx<T> v[EPT];
    if (live) {
#pragma unroll
      for (int k = 0; k < EPT; ++k) {
        const int e = t + k * NT;
        g[k] = gq[(long)cq * H + (e <= M - e ? e : M - e)];
      }
#pragma unroll
      for (int k = 0; k < EPT / 2; ++k) {
        const int e = t + k * NT;
        v[k] = e < N ? col[LdsGridCol<RS>()(e)] : mk(T(0), T(0));
      }
    }
    FftSync<M, E>::stage();
    reg_fft<T, M, -1, true, false, E>(v, col, tws, t, live, LdsGridCol<RS>());
    if (live) {
#pragma unroll
      for (int k = 0; k < EPT; ++k) v[k] = cmul(v[k], mk(T(g[k].x), T(g[k].y)));
    }
    FftSync<M, E>::stage();
    reg_fft<T, M, +1, false, true, E>(v, col, tws, t, live, LdsGridCol<RS>());
    FftSync<M, E>::stage();
    if (live) {
#pragma unroll
      for (int k = 0; k < EPT / 2; ++k) {
        const int e = t + k * NT;
        if (e < N) col[LdsGridCol<RS>()(e)] = v[k];
      }
    }
  }
  __syncthreads();
  // rows: inverse, crop, scale, combine with x
  for (int r0 = 0; r0 < N; r0 += PER) {
    const int r = r0 + l;
    const bool live = r < N;
    cplx<T>* row = buf + r * RS + (r >> 3);
    const long rb = (long)r * N;
    cplx<T> v[EPT], xv[EPT / 2];
    T cv[EPT / 2];
#pragma unroll
    for (int k = 0; k < EPT / 2; ++k) {
      const int e = t + k * NT;
      const bool in = live && e < N;
      xv[k] = in && mode != kModeGreen ? x[rb + e] : mk(T(0), T(0));
      cv[k] = in && mode == kModeAdjoint ? chi[rb + e] : T(1);
    }
    if (live) {
#pragma unroll
      for (int k = 0; k < EPT; ++k) v[k] = row[LdsGridRow()(t + k * NT)];
    }
    FftSync<M, E>::stage();
    reg_fft<T, M, +1, false, true, E>(v, row, tws, t, live, LdsGridRow());
#pragma unroll
    for (int k = 0; k < EPT / 2; ++k) {
      const int e = t + k * NT;
      if (!live || e >= N) continue;
      const cplx<T> g = cscale(v[k], inv);
      cplx<T> o = g;
      if (mode == kModeForward) o = csub(xv[k], g);
      else if (mode == kModeAdjoint) o = csub(xv[k], cscale(g, cv[k]));
      y[rb + e] = o;
    }
  }
}

// Full-size 2-D FFT helpers for the one-off spectrum precompute (FP64).
template <typename T, int M, int SIGN>
__global__ void __launch_bounds__((FftShape<M, kFftE<M>>::WG))
k_fft_rows(cplx<T>* __restrict__ data, int rows, int rows_per_wg, const cplx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* smem = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int NT = FftShape<M, kFftE<M>>::NT;
  constexpr int EPT = FftShape<M, kFftE<M>>::EPT;
  const int t = threadIdx.x % NT, rl = threadIdx.x / NT;
  const int row = blockIdx.x * rows_per_wg + rl;
  const bool live = row < rows;
  FftTwiddles<T, M> tws;
  tws.load(tw, t);
  cplx<T> v[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) v[k] = live ? data[(long)row * M + t + k * NT] : mk(T(0), T(0));
  reg_fft<T, M, SIGN>(v, smem + rl * LdsLen<M>::value, tws, t);
  if (live)
#pragma unroll
    for (int k = 0; k < EPT; ++k) data[(long)row * M + t + k * NT] = v[k];
}

template <typename T, int M, int SIGN>
__global__ void __launch_bounds__((FftShape<M, kFftE<M>>::WG))
k_fft_cols(cplx<T>* __restrict__ data, int cols_per_wg, const cplx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* smem = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int NT = FftShape<M, kFftE<M>>::NT;
  constexpr int EPT = FftShape<M, kFftE<M>>::EPT;
  constexpr int ML = LdsLen<M>::value;
  const int c0 = blockIdx.x * cols_per_wg;
  for (int idx = threadIdx.x; idx < M * cols_per_wg; idx += blockDim.x) {
    const int r = idx / cols_per_wg, c = idx % cols_per_wg;
    smem[c * ML + lpad(r)] = data[(long)r * M + c0 + c];
  }
  __syncthreads();
  const int t = threadIdx.x % NT, cl = threadIdx.x / NT;
  FftTwiddles<T, M> tws;
  tws.load(tw, t);
  cplx<T>* buf = smem + cl * ML;
  cplx<T> v[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) v[k] = buf[lpad(t + k * NT)];
  FftSync<M>::stage();
  reg_fft<T, M, SIGN>(v, buf, tws, t);
  FftSync<M>::stage();
#pragma unroll
  for (int k = 0; k < EPT; ++k) buf[lpad(t + k * NT)] = v[k];
  __syncthreads();
  for (int idx = threadIdx.x; idx < M * cols_per_wg; idx += blockDim.x) {
    const int r = idx / cols_per_wg, c = idx % cols_per_wg;
    data[(long)r * M + c0 + c] = smem[c * ML + lpad(r)];
  }
}

// ---------------------------------------------------------------------------
// Green's-function generators (FP64)
// ---------------------------------------------------------------------------
// Block g[i, j] (i, j < N) of the BTTB generator.
//  kind 0 (the benchmark operator, k0^2 G): off-diagonal kh^2 (i/4) H0(kh rho),
//         self term (i pi ka/2) H1(ka) - 1, ka = kh / sqrt(pi).
//  kind 1 (reference operator, B/MKL_GMRES_test_09122019/source/loop_functions.h:139-142):
//         (i/4) H0(k sqrt((i - sr)^2 + (j - sc)^2)) for every (i, j), the
//         half-cell shift sr = 0.5 (C++ orientation) or sc = 0.5 (Python
//         orientation, B/PyGMRES/GMRES.py:23-27).
__global__ void k_green_block(double2* __restrict__ blk, int N, int kind, double k, double sr,
                              double sc) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= (long)N * N) return;
  const int i = (int)(p / N), j = (int)(p % N);
  double re, im, J0, J1, Y0, Y1;
  if (kind == 0) {
    if (i == 0 && j == 0) {
      const double ka = k / sqrt(CGM_PI);
      bessel01(ka, J0, J1, Y0, Y1);
      re = -0.5 * CGM_PI * ka * Y1 - 1.0;
      im = 0.5 * CGM_PI * ka * J1;
    } else {
      const double rho = sqrt((double)i * i + (double)j * j);
      bessel01(k * rho, J0, J1, Y0, Y1);
      re = -0.25 * k * k * Y0;
      im = 0.25 * k * k * J0;
    }
  } else {
    const double di = i - sr, dj = j - sc;
    bessel01(k * sqrt(di * di + dj * dj), J0, J1, Y0, Y1);
    re = -0.25 * Y0;
    im = 0.25 * J0;
  }
  blk[p] = make_double2(re, im);
}

// Reads the generator out of a (2N-1)^2 embedded array laid out as the
// reference's G_prep (B/MKL_GMRES_test_09122019/source/loop_functions.h:150-163).
__global__ void k_gprep_block(const float2* __restrict__ gprep, double2* __restrict__ blk, int N) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= (long)N * N) return;
  const int i = (int)(p / N), j = (int)(p % N);
  const float2 v = gprep[(long)i * (2 * N - 1) + j];
  blk[p] = make_double2(v.x, v.y);
}

// E[(di mod M), (dj mod M)] = blk[|di|, |dj|] for |di|, |dj| < N, else 0.
__global__ void k_embed(const double2* __restrict__ blk, double2* __restrict__ E, int N, int M) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= (long)M * M) return;
  const int r = (int)(p / M), c = (int)(p % M);
  const int ai = r < N ? r : (r > M - N ? M - r : -1);
  const int aj = c < N ? c : (c > M - N ? M - c : -1);
  E[p] = (ai >= 0 && aj >= 0) ? blk[(long)ai * N + aj] : make_double2(0.0, 0.0);
}

// Quarter of the even-symmetric spectrum, stored column-frequency major:
// gq[c' * (M/2+1) + r'] = Ghat[r', c'].
template <typename G>
__global__ void k_quarter(const double2* __restrict__ E, G* __restrict__ gq, int M) {
  const int H = M / 2 + 1;
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= (long)H * H) return;
  const int cq = (int)(p / H), rq = (int)(p % H);
  const double2 v = E[(long)rq * M + cq];
  G o;
  o.x = v.x;
  o.y = v.y;
  gq[p] = o;
}

// ---------------------------------------------------------------------------
// host-side dispatch over the supported embedding sizes
// ---------------------------------------------------------------------------
#define CGM_FOR_EACH_M(X) \
  X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(768) \
  X(1024) X(1536) X(2048) X(3072) X(4096)

int fft_threads(int M) {
  switch (M) {
#define X(m) case m: return FftShape<m, kFftE<m>>::NT;
    CGM_FOR_EACH_M(X)
#undef X
  }
  return 0;
}

// Threads of one transform in the pass kernels.
int pass_threads(int M, bool fp64) {
  switch (M) {
#define X(m) case m: return fp64 ? FftShape<m, kPassE<double, m>>::NT : FftShape<m, kPassE<float, m>>::NT;
    CGM_FOR_EACH_M(X)
#undef X
  }
  return 0;
}

// Largest work-group (threads) the pass kernels of size M accept.
int pass_max_threads(int M, bool fp64) {
  switch (M) {
#define X(m) \
  case m: return fp64 ? PassWG<double, m, kPassE<double, m>>::value : PassWG<float, m, kPassE<float, m>>::value;
    CGM_FOR_EACH_M(X)
#undef X
  }
  return 0;
}

int choose_embedding(int N) {
  static const int sizes[] = {16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768,
                              1024, 1536, 2048, 3072, 4096};
  for (int s : sizes)
    if (s >= 2 * N - 1) return s;
  return 0;
}

static int groups_for(int M, int target_threads) {
  const int nt = fft_threads(M);
  int g = target_threads / nt;
  return g < 1 ? 1 : g;
}

template <typename T>
int launch_pass1(const Plan& P, hipStream_t st, const cplx<T>* x, cplx<T>* xw, const T* chi,
                 const double* norm_ptr, int mode, cplx<T>* Tm, const cplx<T>* tw, const int* done,
                 int B, const BatchStrides& bs) {
  const int M = P.M, N = P.N;
  if constexpr (sizeof(T) == 4) {
    if (M == 1024 && P.wide1_batch > 0 && B >= P.wide1_batch) {
      constexpr int E = kWideE, R = 256 / FftShape<1024, E>::NT;
      hipLaunchKernelGGL((k_pass1<T, 1024, E>), dim3((N + R - 1) / R, B), dim3(256),
                         R * lds_len(M) * sizeof(cplx<T>), st, x, xw, chi, norm_ptr, mode, Tm, N, R, tw, done, bs);
      return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
    }
  }
  const int rows = P.rows1;
  const int grid = (N + rows - 1) / rows;
  const int threads = rows * pass_threads(M, sizeof(T) == 8);
  const size_t lds = (size_t)rows * lds_len(M) * sizeof(cplx<T>);
  if (threads > pass_max_threads(M, sizeof(T) == 8) || lds > kMaxLds) return CGM_ERROR_UNSUPPORTED;
  switch (M) {
#define X(m)                                                                                 \
  case m:                                                                                    \
    hipLaunchKernelGGL((k_pass1<T, m, kPassE<T, m>>), dim3(grid, B), dim3(threads), lds, st, x, xw, chi,   \
                       norm_ptr, mode, Tm, N, rows, tw, done, bs);                            \
    break;
    CGM_FOR_EACH_M(X)
#undef X
    default: return CGM_ERROR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
}

template <typename T, typename G>
int launch_pass2(const Plan& P, hipStream_t st, cplx<T>* Tm, const G* gq, const cplx<T>* tw,
                 const int* done, int B, const BatchStrides& bs) {
  const int M = P.M, N = P.N;
  if constexpr (sizeof(T) == 4) {
    if (M == 1024 && P.wide2_batch > 0 && B >= P.wide2_batch) {
      constexpr int E = kWideE, C = 256 / FftShape<1024, E>::NT;
      hipLaunchKernelGGL((k_pass2<T, G, 1024, E>), dim3(M / C, B), dim3(C * FftShape<1024, E>::NT),
                         C * lds_len(M) * sizeof(cplx<T>), st, Tm, gq, N, C, tw, done, bs);
      return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
    }
  }
  const int cols = P.cols2;
  const int grid = M / cols;
  const int threads = cols * pass_threads(M, sizeof(T) == 8);
  const size_t lds = (size_t)cols * lds_len(M) * sizeof(cplx<T>);
  if (threads > pass_max_threads(M, sizeof(T) == 8) || lds > kMaxLds || M % cols) return CGM_ERROR_UNSUPPORTED;
  switch (M) {
#define X(m)                                                                                  \
  case m:                                                                                     \
    hipLaunchKernelGGL((k_pass2<T, G, m, kPassE<T, m>>), dim3(grid, B), dim3(threads), lds, st, Tm, gq, N,    \
                       cols, tw, done, bs);                                                   \
    break;
    CGM_FOR_EACH_M(X)
#undef X
    default: return CGM_ERROR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
}

template <typename T>
int launch_pass3(const Plan& P, hipStream_t st, const cplx<T>* Tm, const cplx<T>* x, const T* chi,
                 const cplx<T>* b, cplx<T>* y, int mode, const cplx<T>* tw, const int* done,
                 int B, const BatchStrides& bs) {
  const int M = P.M, N = P.N;
  if constexpr (sizeof(T) == 4) {
    if (M == 1024 && P.wide3_batch > 0 && B >= P.wide3_batch) {
      constexpr int E = kWideE, R = 256 / FftShape<1024, E>::NT;
      hipLaunchKernelGGL((k_pass3<T, 1024, E>), dim3((N + R - 1) / R, B), dim3(256),
                         R * lds_len(M) * sizeof(cplx<T>), st, Tm, x, chi, b, y, mode, N, R,
                         T(1.0 / ((double)M * (double)M)), tw, done, bs);
      return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
    }
  }
  const int rows = P.rows3;
  const int grid = (N + rows - 1) / rows;
  const int threads = rows * pass_threads(M, sizeof(T) == 8);
  const size_t lds = (size_t)rows * lds_len(M) * sizeof(cplx<T>);
  if (threads > pass_max_threads(M, sizeof(T) == 8) || lds > kMaxLds) return CGM_ERROR_UNSUPPORTED;
  const T inv = T(1.0 / ((double)M * (double)M));
  switch (M) {
#define X(m)                                                                                   \
  case m:                                                                                      \
    hipLaunchKernelGGL((k_pass3<T, m, kPassE<T, m>>), dim3(grid, B), dim3(threads), lds, st, Tm, x, chi, b,   \
                       y, mode, N, rows, inv, tw, done, bs);                                   \
    break;
    CGM_FOR_EACH_M(X)
#undef X
    default: return CGM_ERROR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
}

// y = A x, A^T x or G x of B vectors in one launch, where the grid is small
// enough (small_matvec); modes FORWARD, ADJOINT, GREEN.  The embedding has to
// fit the 160 KB of LDS of one work-group.  Within that, one launch is the
// better form at every batch: it moves x, chi and y and nothing else.
template <typename T>
bool small_matvec(const Plan& P) {
  return P.M <= (sizeof(T) == 4 ? 96 : 64);
}
template <typename T, typename G>
int launch_small(const Plan& P, hipStream_t st, const cplx<T>* x, const T* chi, const G* gq, cplx<T>* y, int mode,
                 const cplx<T>* tw, int B, const BatchStrides& bs) {
  const T inv = T(1.0 / ((double)P.M * (double)P.M));
  switch (P.M) {
#define X(m)                                                                                                      \
  case m:                                                                                                         \
    if constexpr (m <= (sizeof(T) == 4 ? 96 : 64))                                                                \
      hipLaunchKernelGGL((k_matvec_small<T, G, m>), dim3(B), dim3(SmallShape<m>::BS), 0, st, x, chi, gq, y, mode, \
                         P.N, inv, tw, bs);                                                                       \
    break;
    X(16) X(24) X(32) X(48) X(64) X(96)
#undef X
    default: return CGM_ERROR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? CGM_SUCCESS : CGM_ERROR_DEVICE;
}
template bool small_matvec<float>(const Plan&);
template bool small_matvec<double>(const Plan&);
template int launch_small<float, float2>(const Plan&, hipStream_t, const float2*, const float*, const float2*, float2*,
                                         int, const float2*, int, const BatchStrides&);
template int launch_small<double, double2>(const Plan&, hipStream_t, const double2*, const double*, const double2*,
                                           double2*, int, const double2*, int, const BatchStrides&);

template int launch_pass1<float>(const Plan&, hipStream_t, const float2*, float2*, const float*,
                                 const double*, int, float2*, const float2*, const int*, int,
                                 const BatchStrides&);
template int launch_pass1<double>(const Plan&, hipStream_t, const double2*, double2*,
                                  const double*, const double*, int, double2*, const double2*,
                                  const int*, int, const BatchStrides&);
template int launch_pass2<float, float2>(const Plan&, hipStream_t, float2*, const float2*,
                                         const float2*, const int*, int, const BatchStrides&);
template int launch_pass2<double, double2>(const Plan&, hipStream_t, double2*, const double2*,
                                           const double2*, const int*, int, const BatchStrides&);
template int launch_pass3<float>(const Plan&, hipStream_t, const float2*, const float2*,
                                 const float*, const float2*, float2*, int, const float2*,
                                 const int*, int, const BatchStrides&);
template int launch_pass3<double>(const Plan&, hipStream_t, const double2*, const double2*,
                                  const double*, const double2*, double2*, int, const double2*,
                                  const int*, int, const BatchStrides&);

int pass_lds_limits(int M) {
  const auto allow = [](const void* f) { return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds); };
  if (M == 4096) {  // a 4096-point FP64 transform
    constexpr int E = kPassE<double, 4096>;
    CGM_HIP(allow((const void*)k_pass1<double, 4096, E>));
    CGM_HIP(allow((const void*)k_pass2<double, double2, 4096, E>));
    CGM_HIP(allow((const void*)k_pass3<double, 4096, E>));
    CGM_HIP(allow((const void*)k_fft_rows<double, 4096, -1>));
    CGM_HIP(allow((const void*)k_fft_cols<double, 4096, -1>));
  }
  return CGM_SUCCESS;
}

int plan_init(Plan& P, int N) {
  P.N = N;
  P.M = choose_embedding(N);
  if (P.M == 0) return CGM_ERROR_UNSUPPORTED;
  const int nt = fft_threads(P.M);
  P.rows1 = groups_for(P.M, 256);
  P.rows3 = P.rows1;
  P.cols2 = groups_for(P.M, 256);
  while (P.M % P.cols2) P.cols2 /= 2;
  if (P.cols2 < 1) P.cols2 = 1;
  P.wide1_batch = P.wide2_batch = P.wide3_batch = 0;
  (void)nt;
  return CGM_SUCCESS;
}

// FP64 spectrum of an N x N generator block in device memory.  Writes the
// complex64 quarter (gq32, may be null) and/or the complex128 quarter
// (gq64, may be null).
int spectrum_from_block(const Plan& P, hipStream_t st, const double2* blk, const double2* tw64,
                        float2* gq32, double2* gq64) {
  const int N = P.N, M = P.M;
  double2* E = nullptr;
  CGM_HIP(hipMallocAsync((void**)&E, sizeof(double2) * (size_t)M * M, st));
  const long MM = (long)M * M;
  hipLaunchKernelGGL(k_embed, dim3((MM + 255) / 256), dim3(256), 0, st, blk, E, N, M);
  const int nt = fft_threads(M);
  const int rows = groups_for(M, 256);
  int cols = rows;
  while (M % cols) cols /= 2;
  const size_t lds = (size_t)rows * lds_len(M) * sizeof(double2);
  switch (M) {
#define X(m)                                                                                   \
  case m:                                                                                      \
    hipLaunchKernelGGL((k_fft_rows<double, m, -1>), dim3((M + rows - 1) / rows),                \
                       dim3(rows * nt), lds, st, E, M, rows, tw64);                             \
    hipLaunchKernelGGL((k_fft_cols<double, m, -1>), dim3(M / cols), dim3(cols * nt),            \
                       (size_t)cols * lds_len(M) * sizeof(double2), st, E, cols, tw64);            \
    break;
    CGM_FOR_EACH_M(X)
#undef X
    default:
      (void)hipFreeAsync(E, st);
      return CGM_ERROR_UNSUPPORTED;
  }
  const int H = M / 2 + 1;
  const long HH = (long)H * H;
  if (gq32) hipLaunchKernelGGL((k_quarter<float2>), dim3((HH + 255) / 256), dim3(256), 0, st, E, gq32, M);
  if (gq64) hipLaunchKernelGGL((k_quarter<double2>), dim3((HH + 255) / 256), dim3(256), 0, st, E, gq64, M);
  CGM_HIP(hipGetLastError());
  CGM_HIP(hipFreeAsync(E, st));
  return CGM_SUCCESS;
}

int green_block(hipStream_t st, double2* blk, int N, int kind, double k, double sr, double sc) {
  const long n = (long)N * N;
  hipLaunchKernelGGL(k_green_block, dim3((n + 255) / 256), dim3(256), 0, st, blk, N, kind, k, sr, sc);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

int gprep_block(hipStream_t st, const float2* gprep, double2* blk, int N) {
  const long n = (long)N * N;
  hipLaunchKernelGGL(k_gprep_block, dim3((n + 255) / 256), dim3(256), 0, st, gprep, blk, N);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

}  // namespace cgm
