// Self-sorting Stockham FFT for one transform of compile-time length M, executed
// by NT = M / EPT threads that each hold EPT elements in registers: element
// t + NT k in register k of thread t, for the input and for the output.  Every
// stage is a DFT over registers; between two stages the data cross threads
// through LDS once.
//
// Stage s with radix R over span Ns (product of earlier radices): butterfly
// j in [0, M/R) reads x[j + r*M/R], multiplies by exp(sign*2*pi*i*r*(j%Ns)/(Ns*R)),
// applies the R-point DFT and writes x[(j/Ns)*Ns*R + j%Ns + r*Ns].  Twiddles
// come from a table tw[q] = exp(-2*pi*i*q/M) built on the host in FP64.
// The unnormalised transform is the one cuFFT computes for the reference
// (B/CUDA_GMRES/Fast_matvec.cuh:13-26).
#pragma once
#include "cgm_common.h"

namespace cgm {

// ---- LDS layout ---------------------------------------------------------------
// Transforms keep one pad element after every 8 in LDS: element e sits at
// e + e/8.  The first radix-8 stage writes x[8j + r] (64-byte lane stride for
// complex64), which without the pad lands every lane of a wave in the same few
// banks; with it the stride is 72 bytes and the writes spread over all banks,
// while stride-1 reads stay contiguous.
__host__ __device__ constexpr int lpad(int e) { return e + (e >> 3); }
template <int M> struct LdsLen {
  static constexpr int value = M + M / 8;
};

// ---- radix plans ------------------------------------------------------------
// E elements per thread.  Radices must divide E, so that every thread owns
// exactly E/R butterflies per stage.
//   powers of two: E = 8 (radices 8, then 4 or 2, or 4 4 in place of 8 2) or 16 (the fewest stages of
//                  at most 16, as even as possible: 128 = 16 8, 1024 = 16 8 8);
//   3 * 2^k:       E = 12 (a radix-12 first stage, then 4s and a 2) or 24 (12,
//                  then 8s and a 4 or 2).
// Fewer stages exchange less through LDS; more elements per thread take more
// registers and leave fewer threads.
template <int M, int E> struct FftShape {
  static constexpr bool pow2 = (M & (M - 1)) == 0;
  static constexpr int EPT = E;
  static constexpr int NT = M / E;
  // work-group size bound used for launch_bounds: groups of transforms fill 256 threads
  static constexpr int WG = NT > 256 ? NT : 256;
  static_assert(pow2 ? (E == 8 || E == 16) : (E == 12 || E == 24), "elements per thread");
};
// Elements per thread without a reason for more.
template <int M> constexpr int kFftE = (M & (M - 1)) == 0 ? 8 : 12;

constexpr int fft_log2(int n) {
  int k = 0;
  while (n > 1) { n >>= 1; ++k; }
  return k;
}
// Radix of stage s (0: there is no such stage).
template <int M, int E> __host__ __device__ constexpr int fft_radix(int s) {
  int n = M;
  if constexpr (E == 16) {
    int left = (fft_log2(M) + 3) / 4;
    for (int k = 0; left > 0; ++k, --left) {
      const int e = (fft_log2(n) + left - 1) / left;
      if (k == s) return 1 << e;
      n >>= e;
    }
    return 0;
  }
  int k = 0;
  if (E == 12 || E == 24) {
    if (s == 0) return 12;
    n /= 12;
    ++k;
  }
  const int top = E == 12 ? 4 : 8;
  if (E == 8) {  // 8s, and two 4s rather than an 8 and a 2
    while (n > 1) {
      const int r = n == 16 ? 4 : n % 8 == 0 ? 8 : n;
      if (k == s) return r;
      n /= r;
      ++k;
    }
    return 0;
  }
  while (n % top == 0 && n > 1) {
    if (k == s) return top;
    n /= top;
    ++k;
  }
  return k == s && n > 1 ? n : 0;  // remainder
}
template <int M, int E> __host__ __device__ constexpr int fft_num_stages() {
  int k = 0;
  while (fft_radix<M, E>(k) > 0) ++k;
  return k;
}

// ---- small DFTs in registers -------------------------------------------------
template <typename T, int SIGN>
__device__ inline void dft2(cplx<T>& a, cplx<T>& b) {
  cplx<T> t = a;
  a = cadd(t, b);
  b = csub(t, b);
}

// multiply by SIGN*i
template <typename T, int SIGN>
__device__ inline cplx<T> mul_si(cplx<T> a) {
  return SIGN < 0 ? mk(a.y, -a.x) : mk(-a.y, a.x);
}

template <typename T, int SIGN>
__device__ inline void dft4(cplx<T>* v) {
  cplx<T> a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
  cplx<T> c = cadd(v[1], v[3]), d = mul_si<T, SIGN>(csub(v[1], v[3]));
  v[0] = cadd(a, c);
  v[2] = csub(a, c);
  v[1] = cadd(b, d);
  v[3] = csub(b, d);
}

template <typename T, int SIGN>
__device__ inline void dft3(cplx<T>* v) {
  const T c1 = T(-0.5);
  const T s1 = T(SIGN) * T(0.86602540378443864676);  // sin(2pi/3) * sign
  cplx<T> a = v[0], b = v[1], c = v[2];
  cplx<T> s = cadd(b, c), d = csub(b, c);
  v[0] = cadd(a, s);
  cplx<T> m = mk(a.x + c1 * s.x, a.y + c1 * s.y);
  // i*s1*d
  cplx<T> r = mk(-s1 * d.y, s1 * d.x);
  v[1] = cadd(m, r);
  v[2] = csub(m, r);
}

template <typename T, int SIGN>
__device__ inline void dft8(cplx<T>* v) {
  // radix-2 split: even/odd 4-point DFTs, then combine with w8^k
  cplx<T> e[4] = {v[0], v[2], v[4], v[6]};
  cplx<T> o[4] = {v[1], v[3], v[5], v[7]};
  dft4<T, SIGN>(e);
  dft4<T, SIGN>(o);
  const T h = T(0.70710678118654752440);
  // w8^1 = (1 + SIGN i)/sqrt2, w8^2 = SIGN i, w8^3 = (-1 + SIGN i)/sqrt2
  cplx<T> o1 = mk(h * (o[1].x - T(SIGN) * o[1].y), h * (o[1].y + T(SIGN) * o[1].x));
  cplx<T> o2 = mul_si<T, SIGN>(o[2]);
  cplx<T> o3 = mk(-h * (o[3].x + T(SIGN) * o[3].y), h * (T(SIGN) * o[3].x - o[3].y));
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[5] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[6] = csub(e[2], o2);
  v[3] = cadd(e[3], o3);
  v[7] = csub(e[3], o3);
}

// 12-point DFT: n = 3 m + p, k = k1 + 4 k2; 4-point DFTs over m, the twiddles
// exp(SIGN 2 pi i p k1 / 12), 3-point DFTs over p.  LO: v[6 ..] are zero and
// not read.
template <typename T, int SIGN, bool LO> __device__ inline void dft12(cplx<T>* v);
// 16-point DFT: n = 4 m + p, k = k1 + 4 k2, the same way with twiddles exp(SIGN 2
// pi i p k1 / 16).  LO: v[8 ..] are zero and not read.
template <typename T, int SIGN, bool LO> __device__ inline void dft16(cplx<T>* v);

template <typename T, int SIGN, int R>
__device__ inline void dft(cplx<T>* v) {
  if constexpr (R == 2) dft2<T, SIGN>(v[0], v[1]);
  else if constexpr (R == 3) dft3<T, SIGN>(v);
  else if constexpr (R == 4) dft4<T, SIGN>(v);
  else if constexpr (R == 8) dft8<T, SIGN>(v);
  else if constexpr (R == 12) dft12<T, SIGN, false>(v);
  else if constexpr (R == 16) dft16<T, SIGN, false>(v);
}

// The same DFTs when the upper half of the inputs, v[R/2 .. R-1], is zero
// (the first stage of a transform of zero-padded data): v[0 .. R/2-1] are
// read, all R outputs written.
template <typename T, int SIGN>
__device__ inline void dft4_lo(cplx<T>* v) {  // v[2] = v[3] = 0
  const cplx<T> a = v[0], d = mul_si<T, SIGN>(v[1]);
  v[2] = csub(a, v[1]);
  v[0] = cadd(a, v[1]);
  v[1] = cadd(a, d);
  v[3] = csub(a, d);
}
template <typename T, int SIGN, bool LO>
__device__ inline void dft12(cplx<T>* v) {
  cplx<T> a[3][4];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
#pragma unroll
    for (int m = 0; m < (LO ? 2 : 4); ++m) a[p][m] = v[3 * m + p];
    if constexpr (LO) dft4_lo<T, SIGN>(a[p]);
    else dft4<T, SIGN>(a[p]);
  }
  const T c = T(0.86602540378443864676), h = T(0.5);  // cos, sin of pi/6
  a[1][1] = cmul(a[1][1], mk(c, T(SIGN) * h));
  a[1][2] = cmul(a[1][2], mk(h, T(SIGN) * c));
  a[1][3] = mul_si<T, SIGN>(a[1][3]);
  a[2][1] = cmul(a[2][1], mk(h, T(SIGN) * c));
  a[2][2] = cmul(a[2][2], mk(-h, T(SIGN) * c));
  a[2][3] = mk(-a[2][3].x, -a[2][3].y);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    cplx<T> b[3] = {a[0][k], a[1][k], a[2][k]};
    dft3<T, SIGN>(b);
    v[k] = b[0];
    v[k + 4] = b[1];
    v[k + 8] = b[2];
  }
}
// a * exp(SIGN 2 pi i Q / 16)
template <typename T, int SIGN, int Q>
__device__ inline cplx<T> rot16(cplx<T> a) {
  constexpr T h = T(0.70710678118654752440);
  constexpr T c1 = T(0.92387953251128675613), s1 = T(0.38268343236508977173);  // cos, sin of pi/8
  if constexpr (Q == 4) {
    return mul_si<T, SIGN>(a);
  } else if constexpr (Q == 2) {
    return mk(h * (a.x - SIGN * a.y), h * (a.y + SIGN * a.x));
  } else if constexpr (Q == 6) {
    return mk(-h * (a.x + SIGN * a.y), h * (SIGN * a.x - a.y));
  } else if constexpr (Q == 1) {
    return cmul(a, mk(c1, SIGN * s1));
  } else if constexpr (Q == 3) {
    return cmul(a, mk(s1, SIGN * c1));
  } else {
    static_assert(Q == 9, "twiddles of the 16-point DFT");
    return cmul(a, mk(-c1, -SIGN * s1));
  }
}

template <typename T, int SIGN, bool LO>
__device__ inline void dft16(cplx<T>* v) {
  cplx<T> a[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
#pragma unroll
    for (int m = 0; m < (LO ? 2 : 4); ++m) a[p][m] = v[4 * m + p];
    if constexpr (LO)
      dft4_lo<T, SIGN>(a[p]);
    else
      dft4<T, SIGN>(a[p]);
  }
  a[1][1] = rot16<T, SIGN, 1>(a[1][1]);
  a[1][2] = rot16<T, SIGN, 2>(a[1][2]);
  a[1][3] = rot16<T, SIGN, 3>(a[1][3]);
  a[2][1] = rot16<T, SIGN, 2>(a[2][1]);
  a[2][2] = rot16<T, SIGN, 4>(a[2][2]);
  a[2][3] = rot16<T, SIGN, 6>(a[2][3]);
  a[3][1] = rot16<T, SIGN, 3>(a[3][1]);
  a[3][2] = rot16<T, SIGN, 6>(a[3][2]);
  a[3][3] = rot16<T, SIGN, 9>(a[3][3]);
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    cplx<T> b[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
    dft4<T, SIGN>(b);
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = b[k2];
  }
}

template <typename T, int SIGN, int R>
__device__ inline void dft_lo(cplx<T>* v) {
  if constexpr (R == 2) {
    v[1] = v[0];
  } else if constexpr (R == 4) {
    dft4_lo<T, SIGN>(v);
  } else if constexpr (R == 12) {
    dft12<T, SIGN, true>(v);
  } else if constexpr (R == 16) {
    dft16<T, SIGN, true>(v);
  } else {
    static_assert(R == 8, "half-zero inputs need an even radix");
    cplx<T> e[4] = {v[0], v[2], v[0], v[0]};  // v[4], v[6] are zero
    cplx<T> o[4] = {v[1], v[3], v[1], v[1]};  // v[5], v[7] are zero
    dft4_lo<T, SIGN>(e);
    dft4_lo<T, SIGN>(o);
    const T h = T(0.70710678118654752440);
    cplx<T> o1 = mk(h * (o[1].x - T(SIGN) * o[1].y), h * (o[1].y + T(SIGN) * o[1].x));
    cplx<T> o2 = mul_si<T, SIGN>(o[2]);
    cplx<T> o3 = mk(-h * (o[3].x + T(SIGN) * o[3].y), h * (T(SIGN) * o[3].x - o[3].y));
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);
    v[7] = csub(e[3], o3);
  }
}

// Twiddles of one thread for every stage with span NS > 1, flattened:
// stage S, butterfly b, r = 1..R-1 at fft_tw_offset<M, E>(S) + b*(R-1) + r-1.
template <int M, int E> __host__ __device__ constexpr int fft_stage_span(int S) {
  int ns = 1;
  for (int s = 0; s < S; ++s) ns *= fft_radix<M, E>(s);
  return ns;
}
template <int M, int E> __host__ __device__ constexpr int fft_tw_offset(int S) {
  int off = 0;
  for (int s = 0; s < S; ++s)
    if (fft_stage_span<M, E>(s) > 1) off += (FftShape<M, E>::EPT / fft_radix<M, E>(s)) * (fft_radix<M, E>(s) - 1);
  return off;
}
template <int M, int E> __host__ __device__ constexpr int fft_tw_count() {
  return fft_tw_offset<M, E>(fft_num_stages<M, E>());
}

template <typename T, int M, int E, int S>
__device__ inline void fft_load_tw(cplx<T>* reg, const cplx<T>* __restrict__ tw, int t) {
  if constexpr (S < fft_num_stages<M, E>()) {
    constexpr int R = fft_radix<M, E>(S);
    constexpr int NS = fft_stage_span<M, E>(S);
    if constexpr (NS > 1) {
      constexpr int NB = FftShape<M, E>::EPT / R;
      constexpr int NT = FftShape<M, E>::NT;
      constexpr int OFF = fft_tw_offset<M, E>(S);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int k = (t + b * NT) % NS;
#pragma unroll
        for (int r = 1; r < R; ++r) reg[OFF + b * (R - 1) + r - 1] = tw[(r * k) * (M / (NS * R))];
      }
    }
    fft_load_tw<T, M, E, S + 1>(reg, tw, t);
  }
}

// A thread's twiddles: registers loaded once per kernel (before the data, so the
// table reads overlap the first global loads) and reused by every forward and
// inverse transform the thread takes part in.  With 12 double elements they
// would take over 100 registers; there they are read from the table (in the L1)
// where they are used (FP64 product at N = 700: 65.6 instead of 72.5 us; with 8
// elements it is the slower form, N = 1024: 86 instead of 83 us).
template <typename T, int M, int E = kFftE<M>> struct FftTwiddles {
  static constexpr bool late = sizeof(T) == 8 && E == 12;
  static constexpr int K = late || fft_tw_count<M, E>() == 0 ? 1 : fft_tw_count<M, E>();
  cplx<T> reg[K];
  const cplx<T>* tab;
  __device__ inline void load(const cplx<T>* __restrict__ tw, int t) {
    if constexpr (late) tab = tw;
    else fft_load_tw<T, M, E, 0>(reg, tw, t);
  }
  // Keeps the compiler from holding table values from one transform to the next.
  __device__ inline void refresh() {
    if constexpr (late) asm volatile("" : "+s"(tab));
  }
  // r-th twiddle of butterfly b of stage S with span NS and radix R
  template <int S, int NS, int R>
  __device__ inline cplx<T> get(int t, int b, int r) const {
    if constexpr (late) return tab[(r * ((t + b * (M / E)) % NS)) * (M / (NS * R))];
    constexpr int OFF = fft_tw_offset<M, E>(S);  // a constant, so that the registers are indexed by constants
    return reg[late ? 0 : OFF + b * (R - 1) + r - 1];
  }
};

// Orders one wave's LDS writes before its later reads (no instruction: the
// wave's LDS accesses complete in issue order; this keeps the compiler from
// moving them across).
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Transforms of at most 64 threads lie within one wave: thread t of the
// transform is lane (t + NT * k) of its wave, since NT is a power of two and
// the groups of NT threads start at multiples of it.  Their stages are ordered
// by the wave's own LDS order and take no work-group barrier: the waves of a
// work-group run through their transforms independently.
template <int M, int E = kFftE<M>> struct FftSync {
  static constexpr bool one_wave = FftShape<M, E>::NT <= 64 && 64 % FftShape<M, E>::NT == 0;
  static __device__ inline void stage() {
    if constexpr (one_wave) wave_lds_sync();
    else __syncthreads();
  }
};

// Where element e of a transform sits in its LDS buffer.
struct LdsRow {
  __device__ inline int operator()(int e) const { return lpad(e); }
};

// Stage S of a transform and the ones after it.  Threads outside the
// transform (active = false) skip the data work but reach the same
// synchronisations: these stay outside any branch, so a wave whose lanes are
// partly inside the transform still executes all of them.
template <typename T, int M, int E, int SIGN, int S, int NS, bool LO, bool HI, typename IX>
__device__ inline void fft_stages(cplx<T>* v, cplx<T>* buf, const FftTwiddles<T, M, E>& tws, int t, bool active, IX at) {
  constexpr int R = fft_radix<M, E>(S);
  constexpr int EPT = E;
  constexpr int NT = FftShape<M, E>::NT;
  constexpr int NB = EPT / R;  // butterflies per thread: j = t + b NT reads registers b + r NB
  constexpr bool lo = LO && S == 0 && R % 2 == 0;
  constexpr bool last = S + 1 == fft_num_stages<M, E>();
  static_assert(!LO || fft_radix<M, E>(0) % 2 == 0, "half-zero inputs need an even first radix");
  static_assert(!HI || fft_radix<M, E>(fft_num_stages<M, E>() - 1) % 2 == 0, "half outputs need an even last radix");
  cplx<T> u[NB][R];
  if (active) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int r = 0; r < (lo ? R / 2 : R); ++r) u[b][r] = v[b + r * NB];
      if constexpr (NS > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cplx<T> w = tws.template get<S, NS, R>(t, b, r);
          if (SIGN > 0) w.y = -w.y;
          u[b][r] = cmul(u[b][r], w);
        }
      }
      if constexpr (lo)
        dft_lo<T, SIGN, R>(u[b]);
      else
        dft<T, SIGN, R>(u[b]);
    }
  }
  if constexpr (last) {
    if (active) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < (HI ? R / 2 : R); ++r) v[b + r * NB] = u[b][r];
    }
  } else {
    if constexpr (S > 0) FftSync<M, E>::stage();  // the previous exchange is read
    if (active) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int j = t + b * NT;
        const int base = (j / NS) * NS * R + j % NS;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[at(base + r * NS)] = u[b][r];
      }
    }
    FftSync<M, E>::stage();
    if (active) {
#pragma unroll
      for (int k = 0; k < EPT; ++k) v[k] = buf[at(t + k * NT)];
    }
    fft_stages<T, M, E, SIGN, S + 1, NS * R, LO, HI>(v, buf, tws, t, active, at);
  }
}

// Length-M transform of v (element t + NT k in v[k]) by threads t in [0, NT),
// in place; buf is M elements of LDS (element e at buf[at(e)]) that no other
// thread uses and that the transform's own threads are done with (FftSync<M, E>::stage()
// before the call if they were not, and before buf is used again after it).
// LO: the upper half of the input is zero (v[EPT/2 ..] is not read).  HI: only
// the outputs below M/2 are formed (v[k], k < EPT/2).
template <typename T, int M, int SIGN, bool LO = false, bool HI = false, int E = kFftE<M>, typename IX = LdsRow>
__device__ inline void reg_fft(cplx<T>* v, cplx<T>* buf, const FftTwiddles<T, M, E>& tws, int t, bool active = true,
                               IX at = IX()) {
  fft_stages<T, M, E, SIGN, 0, 1, LO, HI>(v, buf, tws, t, active, at);
}

}  // namespace cgm
