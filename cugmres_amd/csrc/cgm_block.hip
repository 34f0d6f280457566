// Orthonormalisation of block GMRES on row blocks: W (s x n, s <= 16 right-hand
// sides) against the basis V (k x n), twice (CGS2), and the Cholesky QR of what
// is left, twice (CholQR2).
//
// The reference projects one vector at a time with a dot per basis vector
// (B/CUDA_GMRES/GMRES.cuh:289-303); here the s vectors of a block step share
// every pass over the basis, so the projections are contractions of (k x n) by
// (n x s) and run on the FP32 matrix cores.  Four passes over V per step bound
// it (8 k n bytes each): two projections, two updates.
//
//   k_bp_proj   H = V^H W, FP32 MFMA sums over a chunk of n, FP64 beyond
//   k_bp_red    H over the chunks, in a fixed order; FP64 total of both passes
//   k_bp_upd    W -= (V H)^T; after the second pass also the Gram matrix of W
//   k_bp_chol   FP64 Gram matrix over the work-groups, its Cholesky factor and
//               the inverse of that
//   k_bp_gram   Gram matrix of the once-orthonormalised block (formed in FP64,
//               never stored)
//   k_bp_out    the twice-orthonormalised block, FP64 arithmetic, rounded once
//
// The MFMA used is 16 x 16 x 4 in FP32: lane (a, g) holds A[a][g], B[g][a] and
// D[4 g + r][a].
#include "cgm_internal.h"
#include "cgm_reduce.h"

using namespace cgm;

namespace {

constexpr int kS = 16;         // rows of a block (fewer: the rest is zero)
constexpr int kRows = 64;      // basis rows per work-group of the projection
constexpr int kX = 128;        // cells per work-group of the update
constexpr int kLd = kX + 1;    // LDS row stride of a block's cells
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ inline f4_t mfma(float a, float b, f4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ inline double2 dfma(double2 a, double2 b, double2 c) {  // a b + c
  return make_double2(c.x + a.x * b.x - a.y * b.y, c.y + a.x * b.y + a.y * b.x);
}
__device__ inline double2 dfmac(double2 a, double2 b, double2 c) {  // conj(a) b + c
  return make_double2(c.x + a.x * b.x + a.y * b.y, c.y + a.x * b.y - a.y * b.x);
}

// Partial sums of H[i][c] = sum_x conj(V_i[x]) W_c[x] over chunk blockIdx.x (ch
// cells, a multiple of 128) for the 64 basis rows of blockIdx.y, to
// part[(chunk * kp + i) * 16 + c] (kp: k padded to 64).  Lane (a, g) of a wave
// loads cells 8 h + 2 g, + 1 (h < 4; 64 bytes of a row per load) of basis row a of
// each of four row tiles and of block row a: each is K-value g of an MFMA, so
// nothing is shuffled.  Re = Vr Wr + Vi Wi, Im = Vr Wi - Vi Wr.  Rows from k on repeat row
// k - 1 and are dropped by k_bp_red, block rows from s on are zero.
__global__ void __launch_bounds__(256)
k_bp_proj(const float2* __restrict__ V, const float2* __restrict__ W, long n, int k, int s, int ch, int kp,
          double2* __restrict__ part) {
  __shared__ float red[4][kRows][kS][2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, a = lane & 15, g = lane >> 4;
  const long x0 = (long)blockIdx.x * ch, x1 = x0 + ch < n ? x0 + ch : n;
  const int r0 = blockIdx.y * kRows;
  const float2* vp[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int i = r0 + 16 * t + a;
    vp[t] = V + (long)(i < k ? i : k - 1) * n + 2 * g;
  }
  const float2* wp = W + (long)(a < s ? a : 0) * n + 2 * g;
  f4_t re[4], p[4], q[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) re[t] = p[t] = q[t] = f4_t{0.f, 0.f, 0.f, 0.f};
  f4_t wv[4], vv[4][4];
  const auto load = [&](long x) {
#pragma unroll
    for (int h = 0; h < 4; ++h) wv[h] = *reinterpret_cast<const f4_t*>(wp + x + 8 * h);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int h = 0; h < 4; ++h) vv[t][h] = __builtin_nontemporal_load(reinterpret_cast<const f4_t*>(vp[t] + x + 8 * h));
  };
  long x = x0 + 32 * w;
  if (x < x1) load(x);
  for (; x < x1; x += 128) {
    f4_t wc[4], vc[4][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      wc[h] = a < s ? wv[h] : f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 4; ++t) vc[t][h] = vv[t][h];
    }
    load(x + 128 < x1 ? x + 128 : x);  // the next cells, while these are multiplied
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const float wr = wc[m >> 1][2 * (m & 1)], wi = wc[m >> 1][2 * (m & 1) + 1];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float vr = vc[t][m >> 1][2 * (m & 1)], vi = vc[t][m >> 1][2 * (m & 1) + 1];
        re[t] = mfma(vr, wr, re[t]);
        p[t] = mfma(vr, wi, p[t]);
        q[t] = mfma(vi, wr, q[t]);
        re[t] = mfma(vi, wi, re[t]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      red[w][16 * t + 4 * g + r][a][0] = re[t][r];
      red[w][16 * t + 4 * g + r][a][1] = p[t][r] - q[t][r];
    }
  __syncthreads();
  double2* P = part + ((long)blockIdx.x * kp + r0) * kS;
  for (int e = threadIdx.x; e < kRows * kS; e += 256) {
    const int i = e / kS, c = e % kS;
    double sr = 0.0, sj = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      sr += red[u][i][c][0];
      sj += red[u][i][c][1];
    }
    P[e] = make_double2(sr, sj);
  }
}

// H over the chunks, in four interleaved sums: H32 (kp x 16, zero from k and s
// on) for the update, and H64 (k x s): set by the first pass, added to by the
// second.
__global__ void __launch_bounds__(256)
k_bp_red(const double2* __restrict__ part, int chunks, int k, int s, int kp, float2* __restrict__ H32,
         double2* __restrict__ H64, int second) {
  __shared__ double2 red[4][64];
  const int l = threadIdx.x & 63, sl = threadIdx.x >> 6;
  const int e = blockIdx.x * 64 + l;  // kp is a multiple of 64
  double2 h = make_double2(0.0, 0.0);
#pragma unroll 8
  for (int u = sl; u < chunks; u += 4) {
    const double2 v = part[(long)u * kp * kS + e];
    h.x += v.x;
    h.y += v.y;
  }
  red[sl][l] = h;
  __syncthreads();
  if (sl) return;
  const int i = e / kS, c = e % kS;
  if (i < k && c < s) {
    // as the update takes it
    const float2 f = make_float2((float)((red[0][l].x + red[1][l].x) + (red[2][l].x + red[3][l].x)),
                                 (float)((red[0][l].y + red[1][l].y) + (red[2][l].y + red[3][l].y)));
    double2* o = H64 + (long)i * s + c;
    *o = second ? make_double2(o->x + f.x, o->y + f.y) : make_double2(f.x, f.y);
    H32[e] = f;
  } else {
    H32[e] = make_float2(0.f, 0.f);
  }
}

// H32 (kp x 16) = -Y (k x s, FP64) for the combination U = Y^T V.
__global__ void __launch_bounds__(256)
k_bp_coef(const double2* __restrict__ Y, int k, int s, int kp, float2* __restrict__ H32) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= kp * kS) return;
  const int i = e / kS, c = e % kS;
  float2 h = make_float2(0.f, 0.f);
  if (i < k && c < s) {
    const double2 y = Y[(long)i * s + c];
    h = make_float2((float)-y.x, (float)-y.y);
  }
  H32[e] = h;
}

// Gram partial of the block's kX cells in LDS (rows of kLd): entry (a, b) =
// sum_x conj(b_a[x]) b_b[x].  A thread takes 2 x 2 entries over a quarter of the
// cells (two LDS values per product instead of four); the quarters meet in red.
template <typename C>
__device__ inline void gram_part(const C* blk, double2 (*red)[kS * kS], double2* __restrict__ out) {
  const int q = threadIdx.x >> 6, a = 2 * ((threadIdx.x >> 3) & 7), b = 2 * (threadIdx.x & 7);
  double2 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = make_double2(0.0, 0.0);
#pragma unroll 4
  for (int x = q; x < kX; x += 4) {
    double2 u[2], v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const C cu = blk[(a + i) * kLd + x], cv = blk[(b + i) * kLd + x];
      u[i] = make_double2(cu.x, cu.y);
      v[i] = make_double2(cv.x, cv.y);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = dfmac(u[i], v[j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) red[q][(a + i) * kS + b + j] = acc[i][j];
  __syncthreads();
  const int e = threadIdx.x;
  out[(long)blockIdx.x * kS * kS + e] = make_double2((red[0][e].x + red[1][e].x) + (red[2][e].x + red[3][e].x),
                                                     (red[0][e].y + red[1][e].y) + (red[2][e].y + red[3][e].y));
}

// Out = In - (V H)^T for the kX cells of work-group blockIdx.x (In null: zero).
// D rows are the block's rows, D columns cells: A = H^T from the L2, B = V, 16
// bytes (two cells) of basis row i + g per lane and 32 cells, 128 cells per
// wave.  The four waves take every fourth group of four basis rows, and their
// sums meet in LDS.  GRAM: also the Gram partial of Out.
template <bool GRAM>
__global__ void __launch_bounds__(256)
k_bp_upd(const float2* V, const float2* __restrict__ H32, const float2* In, float2* Out, long n, int k, int s, double2* __restrict__ gpart) {
  __shared__ float red[4][64][64];  // wave, register, lane; then the block's cells
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, a = lane & 15, g = lane >> 4;
  const long x0 = (long)blockIdx.x * kX;
  f4_t acc[4][2][2];  // 32 cells, cell of the pair, re / im
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int e = 0; e < 2; ++e) acc[p][e][0] = acc[p][e][1] = f4_t{0.f, 0.f, 0.f, 0.f};
  const float2* xp = V + x0 + 2 * a;
  const long left = n - x0;  // a multiple of 64
#pragma unroll 2
  for (int i = 4 * w; i < k; i += 16) {
    const int row = i + g < k ? i + g : k - 1;  // H is zero from k on
    const float2 h = H32[(i + g) * kS + a];
    f4_t v[4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
      v[p] = __builtin_nontemporal_load(reinterpret_cast<const f4_t*>(xp + (long)row * n + (32 * p < left ? 32 * p : 0)));
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float vr = v[p][2 * e], vi = v[p][2 * e + 1];
        acc[p][e][0] = mfma(h.x, vr, acc[p][e][0]);
        acc[p][e][1] = mfma(h.x, vi, acc[p][e][1]);
        acc[p][e][0] = mfma(-h.y, vi, acc[p][e][0]);
        acc[p][e][1] = mfma(h.y, vr, acc[p][e][1]);
      }
  }
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[w][((p * 2 + e) * 2 + c) * 4 + r][lane] = acc[p][e][c][r];
  __syncthreads();
  // wave w takes cells x0 + 32 w + 2 a, + 1 of rows 4 g .. 4 g + 3
  f4_t o[4];
  const long x = x0 + 32 * w + 2 * a;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    f4_t d;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int reg = ((w * 2 + (q >> 1)) * 2 + (q & 1)) * 4 + r;
      d[q] = (red[0][reg][lane] + red[1][reg][lane]) + (red[2][reg][lane] + red[3][reg][lane]);
    }
    const int c = 4 * g + r;
    const bool in = c < s && 32 * w < left;
    f4_t v = {0.f, 0.f, 0.f, 0.f};
    if (in && In) v = *reinterpret_cast<const f4_t*>(In + (long)c * n + x);
    o[r] = in ? v - d : f4_t{0.f, 0.f, 0.f, 0.f};
    if (in) *reinterpret_cast<f4_t*>(Out + (long)c * n + x) = o[r];
  }
  if constexpr (GRAM) {
    __syncthreads();
    float2* blk = reinterpret_cast<float2*>(red);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float2* q = blk + (4 * g + r) * kLd + 32 * w + 2 * a;
      q[0] = make_float2(o[r][0], o[r][1]);
      q[1] = make_float2(o[r][2], o[r][3]);
    }
    __syncthreads();
    gram_part(blk, reinterpret_cast<double2(*)[kS * kS]>(reinterpret_cast<char*>(red) + 32768), gpart);
  }
}

// G over the nparts partials in a fixed order, G = (G + G^H) / 2 with the
// identity from s on, G = L L^H, X = inv(conj(L)).  First factorisation: M = X,
// S = L^H.  Second: M = X M, S = L^H S, written to Sout (s x s).  *flag: 1 when a
// pivot is not positive, 2 when the smallest |L_ii|^2 is at most tol times the
// largest diagonal entry of G (M, S then hold no use); kept from the first.
//
// kCholWgs work-groups add up their share of the partials; the last one to
// arrive (its ticket is reset) adds up the shares and factors.  Step q of the
// elimination updates the trailing part of G and of the right-hand side
// (identity, for the inverse) from column q and row q as they stand, so a step
// is one barrier.
constexpr int kCholWgs = 16;
__global__ void __launch_bounds__(256)
k_bp_chol(const double2* __restrict__ gpart, int nparts, int s, double tol, int second, double2* __restrict__ share,
          unsigned* ticket, double2* __restrict__ M, double2* __restrict__ S, double2* __restrict__ Sout,
          double2* __restrict__ flag) {
  __shared__ double2 A[kS][kS + 1], X[kS][kS + 1], L[kS][kS + 1], g[kS * kS];
  const int e = threadIdx.x, i = e >> 4, j = e & 15;
  double2 acc = make_double2(0.0, 0.0);
#pragma unroll 8
  for (int u = blockIdx.x; u < nparts; u += kCholWgs) {
    const double2 v = gpart[(long)u * kS * kS + e];
    acc.x += v.x;
    acc.y += v.y;
  }
  put2(&share[blockIdx.x * kS * kS + e], acc.x, acc.y);
  if (!arrive_last(ticket)) return;
  if (e == 0) reset_ticket(ticket);
  acc = make_double2(0.0, 0.0);
  double2 v[kCholWgs];
#pragma unroll
  for (int u = 0; u < kCholWgs; ++u) v[u] = get2(&share[u * kS * kS + e]);
#pragma unroll
  for (int u = 0; u < kCholWgs; ++u) {
    acc.x += v[u].x;
    acc.y += v[u].y;
  }
  g[e] = acc;
  __syncthreads();
  const double2 t = g[j * kS + i];
  const double2 m1 = second ? M[e] : make_double2(0.0, 0.0), s1 = second ? S[e] : make_double2(0.0, 0.0);
  A[i][j] = i < s && j < s ? make_double2(0.5 * (acc.x + t.x), 0.5 * (acc.y - t.y)) : make_double2(i == j ? 1.0 : 0.0, 0.0);
  X[i][j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
  __syncthreads();
  double dmax = 0.0;
  for (int q = 0; q < s; ++q) dmax = A[q][q].x > dmax ? A[q][q].x : dmax;
  bool bad = false;
  double lmin = __builtin_huge_val();
  for (int q = 0; q < kS; ++q) {
    const double d = A[q][q].x;
    bad |= !(d > 0.0);
    if (q < s && d < lmin) lmin = d;
    const double r = d > 0.0 ? 1.0 / sqrt(d) : 1.0;
    const double2 ai = A[i][q], aj = A[j][q], xq = X[q][j];
    const double2 li = make_double2(ai.x * r, ai.y * r), lj = make_double2(aj.x * r, aj.y * r);
    if (j == q) L[i][q] = i > q ? li : make_double2(i == q && d > 0.0 ? sqrt(d) : 0.0, 0.0);
    if (i > q) {
      if (j > q && i >= j) {  // A[i][j] -= L[i][q] conj(L[j][q])
        A[i][j].x -= li.x * lj.x + li.y * lj.y;
        A[i][j].y -= li.y * lj.x - li.x * lj.y;
      }
      // X[i][j] -= conj(L[i][q]) X[q][j] / L[q][q]
      const double2 x = make_double2(xq.x * r, xq.y * r);
      X[i][j].x -= li.x * x.x + li.y * x.y;
      X[i][j].y -= li.x * x.y - li.y * x.x;
    }
    __syncthreads();
  }
  {  // the rows of the inverse over their pivots
    const double l = L[i][i].x;
    X[i][j] = j <= i ? make_double2(X[i][j].x / l, X[i][j].y / l) : make_double2(0.0, 0.0);
  }
  if (e == 0) {
    const double f = bad ? 1.0 : lmin <= tol * dmax ? 2.0 : 0.0;
    if (!second || flag->x == 0.0) *flag = make_double2(f, 0.0);
  }
  if (!second) {
    M[e] = X[i][j];
    S[e] = j >= i ? make_double2(L[j][i].x, -L[j][i].y) : make_double2(0.0, 0.0);  // L^H
    return;
  }
  __syncthreads();
  A[i][j] = m1;
  __syncthreads();
  double2 m = make_double2(0.0, 0.0), w = make_double2(0.0, 0.0);
  for (int q = 0; q <= i; ++q) m = dfma(X[i][q], A[q][j], m);
  __syncthreads();
  A[i][j] = s1;
  __syncthreads();
  for (int q = i; q < kS; ++q) w = dfma(make_double2(L[q][i].x, -L[q][i].y), A[q][j], w);
  M[e] = m;
  if (i < s && j < s) Sout[i * s + j] = w;
}

// The kX cells of the block at x0, rows from s on zero, into LDS.
__device__ inline void load_block(const float2* __restrict__ W, long n, int s, long x0, float2* blk) {
  for (int e = threadIdx.x; e < kS * kX; e += 256) {
    const int c = e / kX, x = e % kX;
    blk[c * kLd + x] = c < s && x0 + x < n ? W[(long)c * n + x0 + x] : make_float2(0.f, 0.f);
  }
}

// (M W)[c][x] in FP64, M lower triangular.
__device__ inline double2 apply_row(const double2* Ml, const float2* blk, int c, int x) {
  double2 v = make_double2(0.0, 0.0);
  for (int b = 0; b <= c; ++b) {
    const float2 u = blk[b * kLd + x];
    v = dfma(Ml[c * kS + b], make_double2(u.x, u.y), v);
  }
  return v;
}

__global__ void __launch_bounds__(256)
k_bp_gram(const float2* __restrict__ W, long n, int s, const double2* __restrict__ M, double2* __restrict__ gpart) {
  __shared__ float2 blk[kS * kLd];
  __shared__ double2 v1[kS * kLd], red[4][kS * kS];
  __shared__ double2 Ml[kS * kS];
  const long x0 = (long)blockIdx.x * kX;
  Ml[threadIdx.x] = M[threadIdx.x];
  load_block(W, n, s, x0, blk);
  __syncthreads();
  const int c = threadIdx.x >> 4;
#pragma unroll 2
  for (int x = threadIdx.x & 15; x < kX; x += 16) v1[c * kLd + x] = apply_row(Ml, blk, c, x);
  __syncthreads();
  gram_part(v1, red, gpart);
}

__global__ void __launch_bounds__(256)
k_bp_out(const float2* __restrict__ W, long n, int s, const double2* __restrict__ M, float2* __restrict__ Vout) {
  __shared__ float2 blk[kS * kLd];
  __shared__ double2 Ml[kS * kS];
  const long x0 = (long)blockIdx.x * kX;
  Ml[threadIdx.x] = M[threadIdx.x];
  load_block(W, n, s, x0, blk);
  __syncthreads();
  for (int e = threadIdx.x; e < s * kX; e += 256) {
    const int c = e / kX, x = e % kX;
    if (x0 + x >= n) continue;
    const double2 v = apply_row(Ml, blk, c, x);
    Vout[(long)c * n + x0 + x] = make_float2((float)v.x, (float)v.y);
  }
}

// Cells per chunk of the projection: about 64 chunks, or as many as give the
// row groups two work-groups per CU; a multiple of 128.
int proj_chunk(long n, int groups) {
  long want = 512 / groups;
  want = want < 64 ? 64 : want;
  long ch = (n + want - 1) / want;
  ch = (ch + 127) / 128 * 128;
  return (int)ch;
}

int ensure(void** p, size_t* cap, size_t need) {
  if (need <= *cap) return CGM_SUCCESS;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  if (hipMalloc(p, need) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();  // the caller reports it; the next launch's check must not
    cgm_set_last_error("block orthonormalisation: allocation of %zu MiB failed", need >> 20);
    return CGM_ERROR_ALLOC;
  }
  *cap = need;
  return CGM_SUCCESS;
}

}  // namespace

// [H of both passes (k x s); S (s x s); (flag, 0)] -> H.  Workspace per context:
// the projection's and the Gram matrices' partial sums (grown as needed).
extern "C" int cgm_block_orthonormalise(cgm_ctx_t c, const cgm_complex64* basis, int k, cgm_complex64* w,
                                        cgm_complex64* out, int s, long n, double tol, cgm_complex128* h) {
  CGM_CHECK(c && w && out && h && (k == 0 || basis), CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(s >= 1 && s <= kS && k >= 0, CGM_ERROR_INVALID_VALUE, "s=%d outside [1, %d] or k=%d < 0", s, kS, k);
  CGM_CHECK(n > 0 && n % 64 == 0 && ((uintptr_t)basis | (uintptr_t)w | (uintptr_t)out) % 16 == 0,
            CGM_ERROR_UNSUPPORTED, "n=%ld must be a multiple of 64, the rows 16-byte aligned", n);
  CGM_HIP(hipSetDevice(c->device));
  hipStream_t st = c->stream;
  const int kp = (k + kRows - 1) / kRows * kRows, groups = kp / kRows;
  const int ch = k ? proj_chunk(n, groups) : 128, chunks = (int)((n + ch - 1) / ch);
  const int wgs = (int)((n + kX - 1) / kX);
  BlockWs& B = c->blk;
  int rc;
  if ((rc = ensure((void**)&B.part, &B.part_cap, sizeof(double2) * kS * (size_t)(k ? kp : 1) * chunks))) return rc;
  if ((rc = ensure((void**)&B.h32, &B.h32_cap, sizeof(float2) * kS * (size_t)(kp + kRows)))) return rc;
  if ((rc = ensure((void**)&B.gram, &B.gram_cap, sizeof(double2) * kS * kS * (size_t)(wgs + 2 + kCholWgs)))) return rc;
  if (!B.ticket) {
    unsigned* p = nullptr;
    CGM_HIP(hipMalloc((void**)&p, sizeof(unsigned)));
    // cleared before the launches below, whose stream need not wait for the null stream's
    if (hipMemset(p, 0, sizeof(unsigned)) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess) {
      (void)hipFree(p);
      cgm_set_last_error("block orthonormalisation: ticket clear failed");
      return CGM_ERROR_DEVICE;
    }
    B.ticket = p;
  }
  const float2* V = (const float2*)basis;
  float2* W = (float2*)w;
  double2 *H = (double2*)h, *M = B.gram + (size_t)wgs * kS * kS, *S = M + kS * kS,
          *share = S + kS * kS;
  double2 *Sout = H + (long)k * s, *flag = Sout + s * s;
  for (int pass = 0; pass < 2 && k; ++pass) {
    hipLaunchKernelGGL(k_bp_proj, dim3(chunks, groups), dim3(256), 0, st, V, W, n, k, s, ch, kp, B.part);
    hipLaunchKernelGGL(k_bp_red, dim3(kp * kS / 64), dim3(256), 0, st, B.part, chunks, k, s, kp, B.h32, H, pass);
    if (pass == 0)
      hipLaunchKernelGGL((k_bp_upd<false>), dim3(wgs), dim3(256), 0, st, V, B.h32, W, W, n, k, s, B.gram);
    else
      hipLaunchKernelGGL((k_bp_upd<true>), dim3(wgs), dim3(256), 0, st, V, B.h32, W, W, n, k, s, B.gram);
  }
  if (!k) hipLaunchKernelGGL((k_bp_upd<true>), dim3(wgs), dim3(256), 0, st, W, B.h32, W, W, n, 0, s, B.gram);
  hipLaunchKernelGGL(k_bp_chol, dim3(kCholWgs), dim3(256), 0, st, B.gram, wgs, s, tol, 0, share, B.ticket, M, S, Sout,
                     flag);
  hipLaunchKernelGGL(k_bp_gram, dim3(wgs), dim3(256), 0, st, W, n, s, M, B.gram);
  hipLaunchKernelGGL(k_bp_chol, dim3(kCholWgs), dim3(256), 0, st, B.gram, wgs, s, tol, 1, share, B.ticket, M, S, Sout,
                     flag);
  hipLaunchKernelGGL(k_bp_out, dim3(wgs), dim3(256), 0, st, W, n, s, M, (float2*)out);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

// u[c] = sum_i y[i][c] basis[i]: (s x n) from y (k x s).
extern "C" int cgm_block_combine(cgm_ctx_t c, const cgm_complex64* basis, int k, const cgm_complex128* y,
                                 cgm_complex64* u, int s, long n) {
  CGM_CHECK(c && basis && y && u, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(s >= 1 && s <= kS && k >= 1, CGM_ERROR_INVALID_VALUE, "s=%d outside [1, %d] or k=%d < 1", s, kS, k);
  CGM_CHECK(n > 0 && n % 64 == 0 && ((uintptr_t)basis | (uintptr_t)u) % 16 == 0, CGM_ERROR_UNSUPPORTED,
            "n=%ld must be a multiple of 64, the rows 16-byte aligned", n);
  CGM_HIP(hipSetDevice(c->device));
  const int kp = (k + kRows - 1) / kRows * kRows;
  BlockWs& B = c->blk;
  const int rc = ensure((void**)&B.h32, &B.h32_cap, sizeof(float2) * kS * (size_t)(kp + kRows));
  if (rc) return rc;
  hipLaunchKernelGGL(k_bp_coef, dim3((kp * kS + 255) / 256), dim3(256), 0, c->stream, (const double2*)y, k, s, kp, B.h32);
  hipLaunchKernelGGL((k_bp_upd<false>), dim3((unsigned)((n + kX - 1) / kX)), dim3(256), 0, c->stream,
                     (const float2*)basis, B.h32, (const float2*)nullptr, (float2*)u, n, k, s, (double2*)nullptr);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

namespace cgm {
void block_free(BlockWs& B) {
  if (B.part) (void)hipFree(B.part);
  if (B.h32) (void)hipFree(B.h32);
  if (B.gram) (void)hipFree(B.gram);
  if (B.ticket) (void)hipFree(B.ticket);
  B = BlockWs();
}
}  // namespace cgm
