// Fourier-neural-operator (FNO) right preconditioner: BF16 MFMA inference and
// training kernels for gfx950.
//
// The reference has no preconditioner (B/CUDA_GMRES/GMRES.cuh runs plain
// GMRES); this network is the learned extension that flexible GMRES
// (cgm_fgmres) applies to each Krylov vector.  For a unit-norm vector v on the
// N x N grid and the contrast map chi:
//
//   a   = (chi * chi_scale, N Re v, N Im v)                 per cell
//   h0  = a W_in + b_in                                      (3 -> 32 channels)
//   h_{l+1} = act_l( h_l W_l + b_l + K_l(h_l) ),  l = 0..3,  act = GELU (tanh
//             form) for l < 3, identity for l = 3
//   out = h4 W_out + b_out                                   (32 -> 2)
//   P(v) = s_id v + (out_0 + i out_1) / N                    (s_id learned)
//
// K_l is the spectral convolution of an FNO (Li et al., "Fourier neural
// operator for parametric partial differential equations", ICLR 2021) with
// retained row frequencies kx in {0..15, N-16..N-1} and column frequencies
// ky in {0..15}:
//   U[c,kx,ky]  = sum_{x,y} h[x,y,c] e^{-2 pi i (kx x + ky y)/N}
//   V[o,kx,ky]  = sum_c U[c,kx,ky] Wspec[kx,ky,c,o]
//   K(h)[x,y,o] = (1/N^2) sum_{kx,ky} w_ky Re(V[o,kx,ky] e^{2 pi i (kx x + ky y)/N}),
//                 w_0 = 1, w_ky = 2 otherwise (the inverse real FFT of the
//                 truncated spectrum).
// Only 32 column frequencies (cos and -sin of 16 ky) survive, so the column
// transforms are GEMMs against an N x 32 basis F[y,2ky] = cos(2 pi ky y/N),
// F[y,2ky+1] = -sin(2 pi ky y/N), and every layer is
//   row projection : A_x = F^T H_x          per grid row x (K = N, MFMA)
//   k_spectral     : DFT of A along x at the 32 kx and the channel mixing per
//                    mode (FP32)
//   k_invx         : inverse DFT along x (FP32) -> B_x
//   cell GEMM      : h' = act([h, F_y] [W; B_x] + b)  per cell (K = 64, MFMA)
// In the forward pass the row projection of each layer's input runs inside
// the kernel that produces it (k_lift_row, k_cell_row), for one sample the
// inverse x-DFT of each row of layers 0-2 runs in the cell GEMM of that row,
// and the last cell GEMM carries the 32 -> 2 projection (k_cell_proj):
// 1 + 3 x 2 + 3 launches for one sample, 1 + 4 x 3 for more.  h0 is a
// pointwise function of (chi, v): outside training it never reaches global
// memory, and layer 0's cell GEMM lifts its row again.  The
// backward pass has separate kernels (k_back_rows, k_back_cells) with the roles
// transposed.
//
// Activations are BF16, channel-last ([sample][x][y][32], 64 bytes per cell);
// MFMA accumulation, the spectral path and all weight gradients are FP32.
#include <math.h>

#include <vector>

#include "cgm_internal.h"
#include "cgm_reduce.h"

namespace cgm {
namespace fno {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int C = 32;   // channels
constexpr int KY = 16;  // retained column frequencies
constexpr int KX = 32;  // retained row frequencies
constexpr int S = 36;   // LDS row stride (bf16) of a lifted row: 16-bank offset between lane groups
constexpr int kLayerParams = C * C + C + KX * KY * C * C * 2;
constexpr long kOffLayer0 = 4 * C;
constexpr long layer_off(int l) { return kOffLayer0 + (long)l * kLayerParams; }
constexpr long kOffOut = kOffLayer0 + 4L * kLayerParams;
constexpr long kOffSkip = kOffOut + 2 * C + 2;  // weight of the identity path
constexpr long kNumParams = kOffSkip + 1;

__device__ inline bf16x8 ld8(const bf16* p) { return __builtin_bit_cast(bf16x8, *(const u32x4*)p); }
__device__ inline f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ inline void st4(bf16* p, float a, float b, float c, float d) {
  struct __align__(8) Q { bf16 v[4]; } q;
  q.v[0] = (bf16)a;
  q.v[1] = (bf16)b;
  q.v[2] = (bf16)c;
  q.v[3] = (bf16)d;
  *(Q*)p = q;
}

// GELU in its tanh form, 0.5 x (1 + tanh(u)), u = sqrt(2/pi) (x + 0.044715 x^3),
// evaluated as x * sigma(2u) with sigma(t) = 1 / (1 + e^-t) (the same function:
// 0.5 (1 + tanh(u)) = sigma(2u)): e^-2u = 2^(x (kE1 + kE2 x^2)) with the
// constants folded, then the hardware exp2 and reciprocal (v_exp_f32,
// v_rcp_f32, 1 ulp; the activations are stored as BF16).  Seven VALU
// instructions per activation, where an IEEE division alone takes ten; the
// cell GEMM evaluates 32 activations per cell.  Limits: x -> +inf gives
// 2^-inf = 0 and x; x -> -inf gives rcp(inf) = 0 and -0.
constexpr float kG0 = 0.7978845608028654f;  // sqrt(2/pi)
constexpr float kG1 = 0.044715f;
constexpr float kE1 = -2.0 * 0.7978845608028654 * 1.4426950408889634;             // -2 sqrt(2/pi) log2(e)
constexpr float kE2 = -2.0 * 0.7978845608028654 * 1.4426950408889634 * 0.044715;  // kE1 * 0.044715
__device__ inline float sig2u(float x) {
  const float t = x * __builtin_fmaf(x * x, kE2, kE1);
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(t));
}
__device__ inline float gelu(float x) { return x * sig2u(x); }
// d/dx [x sigma(2u)] = sigma + x sigma (1 - sigma) 2u'
__device__ inline float dgelu(float x) {
  const float sg = sig2u(x);
  return sg + x * sg * (1.f - sg) * 2.f * kG0 * (1.f + 3.f * kG1 * x * x);
}

__device__ inline bool skip(const int* done) { return done && *done; }

__device__ const double kOne = 1.0;  // the norm of a vector that needs no scaling

// Gradient of the last activation, dh4[p][c] = d0 W_out[c][0] + d1 W_out[c][1]
// with (d0, d1) = dz[p] / s, at 8 channels c0..c0+7 (w: their 16 entries of
// W_out, from dproj_weights).  The one rounding of dh4: every kernel that
// needs it forms it from the 8 bytes of dz, so its 64 bytes per cell are
// never stored.  One product is rounded before the sum: the first at
// channels 1, 5, ... and from 30 on the second factor's, elsewhere the other
// way round.  The choice decides a BF16 rounding now and then, which the
// layers below amplify to 1e-3 of a weight's gradient: it is fixed, so that
// a training run is reproducible across versions of these kernels.
__device__ inline void dproj_weights(const float* __restrict__ Wout, int c0, float* w) {
#pragma unroll
  for (int k = 0; k < 16; ++k) w[k] = Wout[2 * c0 + k];
  if (c0 + 8 == C) {  // channels 30 and 31 take their factors in the other order
    const float t6 = w[12], t7 = w[14];
    w[12] = w[13];
    w[14] = w[15];
    w[13] = t6;
    w[15] = t7;
  }
}
__device__ inline bf16x8 dproj8(float2 dz, float is, int c0, const float* w) {
  const float d0 = dz.x * is, d1 = dz.y * is;
  const float e0 = c0 + 8 == C ? d1 : d0, e1 = c0 + 8 == C ? d0 : d1;  // channels 6, 7 of the eight
  bf16x8 h;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float a = k < 6 ? d0 : e0, b = k < 6 ? d1 : e1;
    h[k] = (bf16)((k & 3) == 1 ? __builtin_fmaf(a, w[2 * k], b * w[2 * k + 1])
                               : __builtin_fmaf(b, w[2 * k + 1], a * w[2 * k]));
  }
  return h;
}

// Four K values of a column of a row-major BF16 tile in LDS: the 16 lanes of
// a group read four rows of 16 elements (lane j the elements 4 (j % 4).. of
// row j / 4) and lane j receives column j.  Two of these are an MFMA operand
// whose K runs over the tile's rows.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ inline bf16x8 ld_tr(const bf16* p0, const bf16* p1) {
  typedef __attribute__((address_space(3))) s16x4 lds4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p0);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p1);
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Sums of NV values over the 16 lanes whose index e is 0..15 (lane = e ST +
// fixed): each step exchanges one half of the values and keeps the other, NV
// exchanges in all where NV full reductions take 4 NV.  Afterwards v[j], j <
// NV / 16, is the sum of value e NV / 16 + j (NV < 16: v[0] that of value
// e / (16 / NV), in all of its lanes).
template <int NV, int ST, int M = 8>
__device__ inline void lane16_sums(float* v, int e) {
  if constexpr (NV > 1) {
    constexpr int H = NV / 2;
    const bool up = e & M;
#pragma unroll
    for (int k = 0; k < H; ++k) {
      const float give = up ? v[k] : v[k + H], keep = up ? v[k + H] : v[k];
      v[k] = keep + __shfl_xor(give, M * ST, 64);
    }
    if constexpr (M > 1) lane16_sums<H, ST, M / 2>(v, e);
  } else {
    v[0] += __shfl_xor(v[0], M * ST, 64);
    if constexpr (M > 1) lane16_sums<1, ST, M / 2>(v, e);
  }
}

// First kernel of a layer's backward pass, one grid row per iteration:
//   out[r][a][c] = sum_y Xt[a][y] Y[r][y][c]                  (Xt: 32 x N basis)
// and the block's weight-gradient partials (Y = the gradient of the layer's
// pre-activations, Z = the layer's input)
//   part[blk][a][c] = sum_r,y Z[r][y][a] Y[r][y][c],  part[blk][C*C + c] = sum_r,y Y[r][y][c].
// DZ: Y is dh4, formed from dz (dproj8); otherwise Y is read.
//
// Bound by the reads of Y and Z (128 bytes per cell, with DZ 72).  The row
// is staged in LDS row-major, 64 bytes per cell, and both operands whose K
// runs over y come from transposing reads; 8 rows apart, the two 32-byte
// halves of a cell are exchanged, so that the 8 rows a half wave touches lie
// in different banks.  Waves 0-3 hold the four 16 x 16 tiles of out, waves
// 4-7 those of the weight gradient; the next row's NC 16-byte items per
// thread are in flight meanwhile.  NC = ceil(N / 128), in steps 1, 2, 4, 8;
// the 16 rows of Xt a wave needs stay in its registers up to NC = 2
// (beyond, they would leave room for one work-group per CU).  At N = 256, 8
// samples: 16 us (15 with DZ), 4.2 TB/s; with 16-bit LDS reads for the
// operands, one work-group of 4 waves per CU and no loads in flight during
// the products the same work took 38 us.  512 work-groups (two per CU): 1,024
// take 18 us and twice the partials.
template <int NC, bool DZ>
__global__ void __launch_bounds__(512, NC <= 4 ? 4 : 2) k_back_rows(const bf16* __restrict__ Xt, const bf16* __restrict__ Y,
                                                   const float2* __restrict__ dz, const float* __restrict__ Wout,
                                                   float is, const bf16* __restrict__ Z,
                                                   float* __restrict__ out, float* __restrict__ part, int N,
                                                   int rows) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* ly = reinterpret_cast<bf16*>(smem_raw);
  bf16* lz = ly + (long)N * C;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int ta = (w >> 1) & 1, tc = w & 1;
  const bool wz = w >= 4;
  const int items = N * 4;
  const int c8 = (tid & 3) * 8;  // this thread's channels (512 % 4 == 0)
  constexpr bool XR = NC <= 2;
  constexpr int NX = XR ? 4 * NC : 1;  // K steps of 32 held
  bf16x8 xa[NX];
  const bf16* xrow = Xt + (long)(16 * ta + i) * N + 8 * g;
  if (XR) {
#pragma unroll
    for (int u = 0; u < NX; ++u) xa[u] = ld8(xrow + (32 * u < N ? 32 * u : 0));
  }
  float wo[16];
  if (DZ) dproj_weights(Wout, c8, wo);
  u32x4 vy[NC], vz[NC];
  float2 vd[NC];
  auto load = [&](long r) {
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      int q = tid + 512 * k;
      q = q < items ? q : items - 1;
      if (DZ)
        vd[k] = dz[r * N + (q >> 2)];
      else
        vy[k] = *reinterpret_cast<const u32x4*>(Y + r * N * C + (long)q * 8);
      vz[k] = *reinterpret_cast<const u32x4*>(Z + r * N * C + (long)q * 8);
    }
  };
  // operand addresses within a K step of 32 rows (rows y with (y >> 3) & 1 == g & 1)
  const int row8 = (8 * g + (i >> 2)) * C + 4 * (i & 3);
  const bf16* pb = ly + row8 + 16 * (tc ^ (g & 1));
  const bf16* pz = lz + row8 + 16 * (ta ^ (g & 1));
  f32x4 accz = {0.f, 0.f, 0.f, 0.f};
  float accb[8] = {};
  load(blockIdx.x);
  for (int r = blockIdx.x; r < rows; r += gridDim.x) {
    __syncthreads();  // the previous row has been read
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int q = tid + 512 * k;
      if (DZ) vy[k] = __builtin_bit_cast(u32x4, dproj8(vd[k], is, c8, wo));
      if (q < items) {
        const int y = q >> 2, o = y * C + (c8 ^ ((y & 8) << 1));
        *reinterpret_cast<u32x4*>(ly + o) = vy[k];
        *reinterpret_cast<u32x4*>(lz + o) = vz[k];
        const bf16x8 hv = __builtin_bit_cast(bf16x8, vy[k]);
#pragma unroll
        for (int j = 0; j < 8; ++j) accb[j] += (float)hv[j];
      }
    }
    __syncthreads();
    load(r + (int)gridDim.x < rows ? r + gridDim.x : r);
    if (!wz) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      if (XR) {
#pragma unroll
        for (int u = 0; u < NX; ++u)
          if (32 * u < N) acc = mma(xa[u], ld_tr(pb + 32 * u * C, pb + 32 * u * C + 4 * C), acc);
      } else {
        for (int y0 = 0; y0 < N; y0 += 64) {  // N % 64 == 0
          const bf16x8 a0 = ld8(xrow + y0), a1 = ld8(xrow + y0 + 32);
          acc = mma(a0, ld_tr(pb + y0 * C, pb + y0 * C + 4 * C), acc);
          acc = mma(a1, ld_tr(pb + (y0 + 32) * C, pb + (y0 + 32) * C + 4 * C), acc);
        }
      }
      float* o = out + (long)r * C * C;
#pragma unroll
      for (int v = 0; v < 4; ++v) o[(16 * ta + 4 * g + v) * C + 16 * tc + i] = acc[v];
    } else {
#pragma unroll 4
      for (int y0 = 0; y0 < N; y0 += 32)
        accz = mma(ld_tr(pz + y0 * C, pz + y0 * C + 4 * C), ld_tr(pb + y0 * C, pb + y0 * C + 4 * C), accz);
    }
  }
  float* pp = part + (long)blockIdx.x * (C * C + C);
  if (wz) {
#pragma unroll
    for (int v = 0; v < 4; ++v) pp[(16 * ta + 4 * g + v) * C + 16 * tc + i] = accz[v];
  }
  __shared__ float sb[8][C];
  lane16_sums<8, 4>(accb, lane >> 2);
  if (!(lane & 4)) sb[w][c8 + (lane >> 3)] = accb[0];
  __syncthreads();
  if (tid < C) {
    float t = 0.f;
    for (int k = 0; k < 8; ++k) t += sb[k][tid];
    pp[C * C + tid] = t;
  }
}

// ---------------------------------------------------------------------------
// Spectral path of a layer from the row projections to the mixed modes, one
// block per (ky, KG retained kx, sample):
//   U[kxi][ch] = s sum_x (in[b][x][2ky][ch] + i in[b][x][2ky+1][ch]) e^{-2 pi i kx x/N}   (saved to usave)
//   forward : s = 1,            V[kxi][o] = w_ky / N^2 sum_c U[kxi][c] W[kxi][ky][c][o]
//   backward: s = w_ky / N^2,   V[kxi][c] = sum_o conj(W[kxi][ky][c][o]) U[kxi][o]
// (w_0 = 1, else 2).  V goes to vout[b][kxi][ky][ch].
//
// Rows go in pairs: pair p >= 1 is rows (p, N - p), whose twiddles are
// conjugate (kx integer), so with P = A_x + A_{N-x}, M = A_x - A_{N-x} and
// e = e^{2 pi i kx x/N} = c + is the pair adds c P - i s M (half the products
// of two rows); pair 0 is rows 0 and N/2 (twiddles 1 and (-1)^kx = (-1)^kxi:
// P at even kxi, M at odd).  32 pairs make a chunk; the sums of the chunks
// are formed by separate threads and added in order, so a sum does not depend
// on KG, which is chosen by the number of blocks.  Sums and products are
// written out as fused or not: every KG rounds alike.
//
// Bound by latencies (the loads of the block's 256 bytes of each row, then a
// chain of 32 pairs, then the mixing), so 512 threads take CP chunks at once:
// thread (chunk, kp, cp) holds RK frequencies x 2 channels.  With 8 and 16
// frequencies CP is 4; five and six chunks (N = 320, 384) take 768 threads
// and CP = 6 (SIX) instead of a second round for the fifth.  One sample of
// N = 512 takes 7.4 us, 8 of N = 256 10.1 (11.1 backward); a transform that
// left its chunks' partial sums to a mixing kernel took 5.0 + 4.0 and
// 7.0 + 5.5 (7.1), and a launch more.
constexpr int kPairs = 32;  // row pairs per chunk
template <int KG, bool SIX = false>
struct SpecShape {
  static constexpr int RK = KG >= 16 ? 2 : 1;   // frequencies per thread
  static constexpr int TPC = KG / RK * 16;      // threads per chunk
  // chunks at once: 512 threads' (at most 8: 128 KiB of P and M), or six
  static constexpr int CP = SIX ? 6 : 512 / TPC < 8 ? 512 / TPC : 8;
  static constexpr int NTHR = SIX ? 6 * TPC : 512;
  static size_t lds(int N) {
    const int nch = N / 64, cp = nch < CP ? nch : CP;
    return (size_t)cp * kPairs * C * 2 * sizeof(float2) + (size_t)KG * (cp * kPairs + 1) * sizeof(float2) +
           (size_t)nch * KG * C * sizeof(float2);
  }
};
template <int KG, bool BWD, bool SIX>
__global__ void __launch_bounds__((SpecShape<KG, SIX>::NTHR)) k_spectral(const float* __restrict__ in, const float2* __restrict__ Ex,
                                                  const float2* __restrict__ W, float2* __restrict__ usave,
                                                  float2* __restrict__ vout, int N, const int* done) {
#pragma clang fp contract(off)
  if (skip(done)) return;
  typedef SpecShape<KG, SIX> Sh;
  constexpr int RK = Sh::RK, TPC = Sh::TPC, CP = Sh::CP, NTHR = Sh::NTHR;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int nch = N / 64, ncp = nch < CP ? nch : CP;
  float2* sp = reinterpret_cast<float2*>(smem_raw);  // [chunk pair][C]
  float2* sm = sp + ncp * kPairs * C;
  float2* part = sm + ncp * kPairs * C;               // [chunk][KG][C]
  float2* se = part + nch * KG * C;                   // [KG][ncp kPairs + 1]
  const int els = ncp * kPairs + 1;
  const int ky = blockIdx.x, k0 = blockIdx.y * KG, b = blockIdx.z;
  const int tid = threadIdx.x;
  // this thread's output of the mixing
  const int kl = tid >> 5, ch = tid & 31, kxi = k0 + kl;
  const bool mixes = tid < KG * C;
  const float2* Wm = W + (long)((mixes ? kxi : k0) * KY + ky) * C * C;
  const int cl = tid / TPC, kp = tid % TPC / 16, cp = tid & 15;
  const float sc = BWD ? (ky == 0 ? 1.f : 2.f) / ((float)N * (float)N) : 1.f;
  auto stage = [&](int g0) {  // P, M and the twiddles of the group's chunks to LDS
    const int pg = g0 * kPairs;                                   // first pair of the group
    const int np = (nch - g0 < CP ? nch - g0 : CP) * kPairs;      // its pairs
    constexpr int NI = CP * kPairs * C / 4 / NTHR;  // items of 4 channels of a pair per thread
    float4 u1[NI][2], u2[NI][2];
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      if (NTHR / 8 * k >= np) break;
      int pl = (tid + NTHR * k) >> 3;
      pl = pl < np ? pl : np - 1;
      const int c4 = (tid & 7) * 4, x = pg + pl, x2 = x == 0 ? N / 2 : N - x;
      const float* r1 = in + ((long)(b * N + x) * C + 2 * ky) * C + c4;
      const float* r2 = in + ((long)(b * N + x2) * C + 2 * ky) * C + c4;
      u1[k][0] = *reinterpret_cast<const float4*>(r1);
      u1[k][1] = *reinterpret_cast<const float4*>(r1 + C);
      u2[k][0] = *reinterpret_cast<const float4*>(r2);
      u2[k][1] = *reinterpret_cast<const float4*>(r2 + C);
    }
    // twiddles: 16 groups of 32 of the first 512 threads, frequency kq, 32 pairs per item
    constexpr int NE = KG * CP * kPairs / 512, SE = 16 / KG * kPairs;
    const int kq = (tid >> 5) % KG, pe = (tid >> 5) / KG * kPairs + (tid & 31);
    float2 ev[NE];
#pragma unroll
    for (int k = 0; k < NE; ++k) ev[k] = Ex[(long)(k0 + kq) * N + pg + (pe + SE * k < np ? pe + SE * k : 0)];
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int pl = (tid + NTHR * k) >> 3, c4 = (tid & 7) * 4;
      if (pl >= np) break;
      const float4 a = u1[k][0], ai = u1[k][1], d = u2[k][0], di = u2[k][1];
      float4* p4 = reinterpret_cast<float4*>(sp + pl * C + c4);
      float4* m4 = reinterpret_cast<float4*>(sm + pl * C + c4);
      p4[0] = make_float4(a.x + d.x, ai.x + di.x, a.y + d.y, ai.y + di.y);
      p4[1] = make_float4(a.z + d.z, ai.z + di.z, a.w + d.w, ai.w + di.w);
      m4[0] = make_float4(a.x - d.x, ai.x - di.x, a.y - d.y, ai.y - di.y);
      m4[1] = make_float4(a.z - d.z, ai.z - di.z, a.w - d.w, ai.w - di.w);
    }
#pragma unroll
    for (int k = 0; k < NE; ++k)
      if ((NTHR == 512 || tid < 512) && pe + SE * k < np) se[kq * els + pe + SE * k] = ev[k];
  };
  auto transform = [&](int g0) {
    const int np = (nch - g0 < CP ? nch - g0 : CP) * kPairs;
    if (cl < CP && cl * kPairs < np) {
      const float2* P = sp + cl * kPairs * C + cp;
      const float2* M = sm + cl * kPairs * C + cp;
      const float2* E = se + RK * kp * els + cl * kPairs;
      float2 acc[RK][2] = {};
      auto add = [&](int pl) {
#pragma unroll
        for (int a = 0; a < RK; ++a)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const float2 e = E[a * els + pl], p = P[pl * C + 16 * c], m = M[pl * C + 16 * c];
            acc[a][c].x = acc[a][c].x + __builtin_fmaf(e.x, p.x, e.y * m.y);  // c P - i s M
            acc[a][c].y = acc[a][c].y + __builtin_fmaf(e.x, p.y, -(e.y * m.x));
          }
      };
      if (g0 + cl == 0) {  // rows 0 and N/2: P at even kxi, M at odd
#pragma unroll
        for (int a = 0; a < RK; ++a)
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[a][c] = (RK * kp + a) & 1 ? M[16 * c] : P[16 * c];
      } else {
        add(0);
      }
#pragma unroll 8
      for (int pl = 1; pl < kPairs; ++pl) add(pl);
#pragma unroll
      for (int a = 0; a < RK; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          part[((g0 + cl) * KG + RK * kp + a) * C + cp + 16 * c] = make_float2(acc[a][c].x * sc, acc[a][c].y * sc);
    }
  };
  stage(0);
  // this thread's 32 weights of the mixing, in flight during the transform
  // (forward: a column of the mode's matrix, coalesced over ch)
  float2 wv[C];
  if (!BWD) {
#pragma unroll
    for (int c = 0; c < C; ++c) wv[c] = Wm[c * C + ch];
  } else {
    const float4* wr = reinterpret_cast<const float4*>(Wm + ch * C);
#pragma unroll
    for (int c = 0; c < C / 2; ++c) {
      const float4 q = wr[c];
      wv[2 * c] = make_float2(q.x, q.y);
      wv[2 * c + 1] = make_float2(q.z, q.w);
    }
  }
  __syncthreads();
  transform(0);
  for (int g0 = CP; g0 < nch; g0 += CP) {
    __syncthreads();
    stage(g0);
    __syncthreads();
    transform(g0);
  }
  __syncthreads();
  float2* su = sp;  // [KG][C]
  const long slot = (((long)b * KX + kxi) * KY + ky) * C + ch;
  if (mixes) {
    float2 u = make_float2(0.f, 0.f);
    for (int k = 0; k < nch; ++k) {
      const float2 t = part[(k * KG + kl) * C + ch];
      u.x = u.x + t.x;
      u.y = u.y + t.y;
    }
    su[kl * C + ch] = u;
    if (usave) usave[slot] = u;
  }
  __syncthreads();
  if (!mixes) return;
  float2 v = make_float2(0.f, 0.f);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float2 u = su[kl * C + c], w = wv[c];
    if (!BWD) {
      v.x = v.x + __builtin_fmaf(u.x, w.x, -(u.y * w.y));
      v.y = v.y + __builtin_fmaf(u.y, w.x, u.x * w.y);
    } else {  // conj(w) u
      v.x = v.x + __builtin_fmaf(w.x, u.x, w.y * u.y);
      v.y = v.y + __builtin_fmaf(w.x, u.y, -(w.y * u.x));
    }
  }
  if (!BWD) {
    const float so = (ky == 0 ? 1.f : 2.f) / ((float)N * (float)N);
    v.x *= so;
    v.y *= so;
  }
  vout[slot] = v;
}

// Inverse DFT along x, XP row pairs of one sample per block (thread = (ky, ch)):
//   out[b][x][ch][2ky], [2ky+1] = Re, Im of sum_kxi V[kxi][ky][ch] e^{+2 pi i kx x/N}   (BF16)
// Rows x and N - x have conjugate twiddles (kx integer), so with V = a + ib,
// e = c + is and the sums S1 = sum a c, S2 = sum b s, S3 = sum a s,
// S4 = sum b c (four products per mode for two rows):
//   B_x = (S1 - S2) + i (S3 + S4),  B_{N-x} = (S1 + S2) + i (S4 - S3).
// Pair p >= 1 is rows (p, N - p); pair 0 is rows 0 and N/2, whose twiddles
// are 1 and (-1)^kx = (-1)^kxi (N even, kx = kxi or N - 32 + kxi).  The
// block's 2 XP x 32 x 32 outputs are assembled in LDS, where the 16-byte
// chunk j of channel ch is at j ^ (ch / 4 % 4) (a wave's writes, one word per
// channel, then touch 32 banks and not 4), and leave as 16-byte stores of
// whole 2 KiB rows.  Every block reads its sample's 128 KiB of modes, so few
// blocks are better as long as every CU has one (N = 256, 8 samples: XP 4 takes
// 6.8 us; XP 8, half the CUs, and unswizzled 2-byte LDS writes 10.2).
template <int XP>
__global__ void __launch_bounds__(512) k_invx(const float2* __restrict__ V, bf16* __restrict__ out,
                                              const float2* __restrict__ Ex, int N, const int* done) {
  if (skip(done)) return;
  __shared__ float2 se[XP][KX];
  __shared__ __align__(16) unsigned int lt[2 * XP][C * C / 2];  // pairs (2ky, 2ky + 1)
  const int p0 = blockIdx.x * XP, b = blockIdx.z;
  const int tid = threadIdx.x;
  if (tid < XP * KX) {
    const int q = tid / XP, pl = tid % XP;
    se[pl][q] = Ex[(long)q * N + p0 + pl];
  }
  const int ch = tid & 31, ky = tid >> 5;
  const int slot = ch * (C / 2) + (ky ^ (((ch >> 2) & 3) << 2));
  auto pack = [](float re, float im) {
    struct P2 { bf16 v[2]; } p{{(bf16)re, (bf16)im}};
    return __builtin_bit_cast(unsigned int, p);
  };
  float2 vq[KX];
#pragma unroll
  for (int q = 0; q < KX; ++q) vq[q] = V[(((long)b * KX + q) * KY + ky) * C + ch];
  __syncthreads();
#pragma unroll 2
  for (int pl = 0; pl < XP; ++pl) {
    float s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f;
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const float2 e = se[pl][q];
      s1 += vq[q].x * e.x;
      s2 += vq[q].y * e.y;
      s3 += vq[q].x * e.y;
      s4 += vq[q].y * e.x;
    }
    lt[pl][slot] = pack(s1 - s2, s3 + s4);
    if (p0 + pl > 0) {
      lt[XP + pl][slot] = pack(s1 + s2, s4 - s3);
    } else {  // row N/2
      float t1 = 0.f, t2 = 0.f;
#pragma unroll
      for (int q = 0; q < KX; q += 2) {
        t1 += vq[q].x - vq[q + 1].x;
        t2 += vq[q].y - vq[q + 1].y;
      }
      lt[XP][slot] = pack(t1, t2);
    }
  }
  __syncthreads();
  // staged row r: x = p0 + r (r < XP), else N - (p0 + r - XP), pair 0's N/2
  const u32x4* src = reinterpret_cast<const u32x4*>(&lt[0][0]);
  for (int q = tid; q < 2 * XP * C * C / 8; q += 512) {
    const int r = q / (C * C / 8), pl = r < XP ? r : r - XP;
    const int x = r < XP ? p0 + pl : (p0 + pl == 0 ? N / 2 : N - p0 - pl);
    reinterpret_cast<u32x4*>(out + ((long)b * N + x) * C * C)[q - r * (C * C / 8)] = src[q ^ ((q >> 4) & 3)];
  }
}

// Spectral weight gradients of the four layers (blockIdx.y), one mode per block:
//   G[kxi][ky][c][o] = sum_b conj(U[b][kxi][ky][c]) dV[b][kxi][ky][o].
// Bound by the 4.2 MB a layer writes; one launch for the four layers, after
// the last of them has its dV (10 us for 8 samples, four launches of a
// thread per output 29).  A thread holds 2 x 2 outputs.
struct SpecGrads {
  const float2* U[4];
  const float2* dV[4];
  float2* G[4];
};
__global__ void __launch_bounds__(256) k_specgrad(SpecGrads t, int B) {
  const int mode = blockIdx.x, l = blockIdx.y;  // kxi * KY + ky
  const int o0 = (threadIdx.x & 15) * 2, c0 = (threadIdx.x >> 4) * 2;
  const float2* U = t.U[l] + (long)mode * C + c0;
  const float2* dV = t.dV[l] + (long)mode * C + o0;
  constexpr long kS = (long)KX * KY * C;  // one sample's modes
  float4 acc[2] = {};
  auto add = [&](const float4& u, const float4& d) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float ux = k ? u.z : u.x, uy = k ? u.w : u.y;
      acc[k].x += ux * d.x + uy * d.y;
      acc[k].y += ux * d.y - uy * d.x;
      acc[k].z += ux * d.z + uy * d.w;
      acc[k].w += ux * d.w - uy * d.z;
    }
  };
  int b = 0;
  for (; b + 8 <= B; b += 8) {
    float4 u[8], d[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      u[k] = *reinterpret_cast<const float4*>(U + (b + k) * kS);
      d[k] = *reinterpret_cast<const float4*>(dV + (b + k) * kS);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) add(u[k], d[k]);
  }
  for (; b < B; ++b)
    add(*reinterpret_cast<const float4*>(U + b * kS), *reinterpret_cast<const float4*>(dV + b * kS));
  // 8-byte stores: grad is only required to be aligned to its elements
  float2* G = t.G[l] + ((long)mode * C + c0) * C + o0;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    G[k * C] = make_float2(acc[k].x, acc[k].y);
    G[k * C + 1] = make_float2(acc[k].z, acc[k].w);
  }
}

// ---------------------------------------------------------------------------
// Per-cell GEMM of the backward pass (layers 3-1), K = 64:
//   out[p][o] = (sum_c P[p][c] A[o][c] + sum_k Q[y][k] R[b][x][o][k]) GELU'(aux[p][o])
// DZ: P is dh4, formed from dz (dproj8); otherwise P is read.  The product is
// formed transposed (rows = output channels, columns = 16 cells) so that lane
// l holds 4 consecutive channels of cell l % 16 in both the B operand and the
// accumulator.  One wave covers 64 consecutive cells of a grid row: bound by
// the 192 bytes per cell read and written (DZ: 136), so every operand of the
// wave is in flight before its first product (21 and 17 us at N = 256, 8
// samples: 4.8 and 4.2 TB/s).
template <bool DZ>
__global__ void __launch_bounds__(256) k_back_cells(const bf16* __restrict__ P, const float2* __restrict__ dz,
                                                    const float* __restrict__ Wout, float is,
                                                    const bf16* __restrict__ Q, const bf16* __restrict__ A,
                                                    const bf16* __restrict__ R, const bf16* __restrict__ aux,
                                                    bf16* __restrict__ out, int N) {
  // each wave stages its 16-cell tile (16 x 32 BF16, rows padded to 80 B) so
  // that every lane stores 16 contiguous bytes and a wave 1 KiB at once
  __shared__ __align__(16) bf16 stage[4][16][40];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const long wv = (long)blockIdx.x * 4 + w;  // every block is full: waves % 4 == 0
  const int segs = N / 64;
  const long bx = wv / segs;  // sample * N + x
  const int y0 = (int)(wv % segs) * 64;
  const int i = lane & 15, g = lane >> 4;
  const int rrow = lane >> 2, rcol = (lane & 3) * 8;
  bf16x8 bpt[4], bqt[4];
  float2 vd[4];
  u32x2 ax[4][2];  // 4 channels of aux per accumulator
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int y = y0 + 16 * t + i;
    const long p = bx * N + y;
    if (DZ)
      vd[t] = dz[p];
    else
      bpt[t] = ld8(P + p * C + 8 * g);
    bqt[t] = ld8(Q + (long)y * C + 8 * g);
#pragma unroll
    for (int to = 0; to < 2; ++to) ax[t][to] = *reinterpret_cast<const u32x2*>(aux + p * C + 16 * to + 4 * g);
  }
  bf16x8 aw[2], ar[2];
#pragma unroll
  for (int to = 0; to < 2; ++to) {
    aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
    ar[to] = ld8(R + (bx * C + 16 * to + i) * C + 8 * g);
  }
  if (DZ) {
    float wo[16];
    dproj_weights(Wout, 8 * g, wo);
#pragma unroll
    for (int t = 0; t < 4; ++t) bpt[t] = dproj8(vd[t], is, 8 * g, wo);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int to = 0; to < 2; ++to) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = mma(aw[to], bpt[t], acc);
      acc = mma(ar[to], bqt[t], acc);
      struct Q4 { bf16 v[4]; };
      const Q4 x = __builtin_bit_cast(Q4, ax[t][to]);
      st4(&stage[w][i][16 * to + 4 * g], acc[0] * dgelu((float)x.v[0]), acc[1] * dgelu((float)x.v[1]),
          acc[2] * dgelu((float)x.v[2]), acc[3] * dgelu((float)x.v[3]));
    }
    // the stage is the wave's own: LDS operations of a wave run in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    *(u32x4*)(out + (bx * N + y0 + 16 * t + rrow) * C + rcol) = *(const u32x4*)&stage[w][rrow][rcol];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// The same GEMM at layer 0 (no activation below it) with the lift's
// gradient.  dh0 is rounded to BF16 as an activation gradient is, but not
// stored: the lift needs only
//   part[blk] = (sum_p a_k dh0[p][c]  [k][c],  sum_p dh0[p][c])
// with (a_0, a_1, a_2) = (chi chi_scale, s Re v, s Im v).  Waves step over
// the 64-cell segments of all samples; a lane holds 8 channels of its cells
// in 32 sums, joined across the block at the end.  12 us at N = 256, 8
// samples; storing dh0 and a second kernel that read it took 30.
__global__ void __launch_bounds__(256) k_back_lift(const bf16* __restrict__ P, const bf16* __restrict__ Q,
                                                   const bf16* __restrict__ A, const bf16* __restrict__ R,
                                                   const float* __restrict__ chi, float chi_scale,
                                                   const float2* __restrict__ v, float s,
                                                   float* __restrict__ part, int N, long nseg) {
  __shared__ float red[4][4 * C];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int segs = N / 64;
  const int i = lane & 15, g = lane >> 4;
  bf16x8 aw[2];
#pragma unroll
  for (int to = 0; to < 2; ++to) aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
  float sum[32] = {};  // [a_0, a_1, a_2, 1][8 channels]
  for (long wv = (long)blockIdx.x * 4 + w; wv < nseg; wv += (long)gridDim.x * 4) {
    const long bx = wv / segs;  // sample * N + x
    const int y0 = (int)(wv - bx * segs) * 64;
    bf16x8 bpt[4], bqt[4], ar[2];
    float cv[4];
    float2 xv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int y = y0 + 16 * t + i;
      const long p = bx * N + y;
      bpt[t] = ld8(P + p * C + 8 * g);
      bqt[t] = ld8(Q + (long)y * C + 8 * g);
      cv[t] = chi[p];
      xv[t] = v[p];
    }
#pragma unroll
    for (int to = 0; to < 2; ++to) ar[to] = ld8(R + (bx * C + 16 * to + i) * C + 8 * g);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float a[3] = {cv[t] * chi_scale, xv[t].x * s, xv[t].y * s};
#pragma unroll
      for (int to = 0; to < 2; ++to) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mma(aw[to], bpt[t], acc);
        acc = mma(ar[to], bqt[t], acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float d = (float)(bf16)acc[q];
#pragma unroll
          for (int k = 0; k < 3; ++k) sum[8 * k + 4 * to + q] += a[k] * d;
          sum[24 + 4 * to + q] += d;
        }
      }
    }
  }
  lane16_sums<32, 1>(sum, i);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int k = (2 * i + j) >> 3, q = (2 * i + j) & 7;
    red[w][k * C + 16 * (q >> 2) + 4 * g + (q & 3)] = sum[j];
  }
  __syncthreads();
  if (tid < 4 * C)
    part[(long)blockIdx.x * 4 * C + tid] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
}

// ---------------------------------------------------------------------------
// Forward-pass kernels that own whole grid rows, so that the row projection of
// the activations they produce (the first step of the next layer's spectral
// convolution) runs on the row while it is still in LDS:
//   k_lift_row  : lift of one row, then A_x = F^T H0_x
//   k_cell_row  : B_x of the row, cell GEMM + GELU of the row (layers 0-2),
//                 then A_x = F^T H'_x
//   k_cell_proj : cell GEMM of layer 3 with the 32 -> 2 projection and the
//                 identity path, z = s_id v + (h4 W_out + b_out) / s
// The row kernels stage the row they project channel-major, [c][y] BF16 with
// row stride basis_ld(N) (the K = y operand of the projection is then 16
// contiguous bytes per lane), and the projection basis F^T likewise.

// Row stride (BF16) of the channel-major row and of the projection basis F^T
// staged in LDS by the row kernels: 16 bytes of padding move row a + 1 four
// banks on, so the 16 rows an MFMA operand read touches fall in different
// banks.
__host__ __device__ constexpr int basis_ld(int N) { return N + 8; }
// LDS bytes of the forward row kernels: the basis and the channel-major row
// or (layer 0's cell GEMM) the row as [y][S].
inline size_t row_kernel_lds(int N) {
  const size_t t = (size_t)C * basis_ld(N) * sizeof(bf16), r = (size_t)N * S * sizeof(bf16);
  return t + (t > r ? t : r);
}

// F^T (32 x N, global) to LDS with row stride basis_ld(N), 16 bytes per item,
// four items per thread in flight together (the loads are unconditional, on
// a clamped item, so that no branch waits for one load before the next is
// issued).
template <int NT>
__device__ inline void basis_to_lds(const bf16* __restrict__ Xt, bf16* lb, int N, int tid = threadIdx.x) {
  const int per_row = N / 8, items = C * per_row;
  u32x4 v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int q = tid + k * NT;
    q = q < items ? q : items - 1;
    const int a = q / per_row, y8 = (q - a * per_row) * 8;
    v[k] = *reinterpret_cast<const u32x4*>(Xt + (long)a * N + y8);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int q = tid + k * NT;
    if (q < items) {
      const int a = q / per_row, y8 = (q - a * per_row) * 8;
      *reinterpret_cast<u32x4*>(lb + a * basis_ld(N) + y8) = v[k];
    }
  }
  for (int q = tid + 4 * NT; q < items; q += NT) {  // N > 16 NT / C only
    const int a = q / per_row, y8 = (q - a * per_row) * 8;
    *reinterpret_cast<u32x4*>(lb + a * basis_ld(N) + y8) = *reinterpret_cast<const u32x4*>(Xt + (long)a * N + y8);
  }
}

// A_x = F^T H_x from the row staged channel-major in LDS (lt[c][y], row
// stride basis_ld(N): the B operand is one 16-byte read), F^T read with row
// stride ldx (from global memory or LDS).  NW waves: wave w owns output tile
// (a-tile (w >> 1) & 1, c-tile w & 1); with NW = 8 waves w and w + 4 split K
// in halves and the upper half adds into the lower through red.
template <int NW>
__device__ inline void row_project(const bf16* __restrict__ Xt, int ldx, const bf16* lt, int N,
                                   float* __restrict__ o, float* red, int tid = threadIdx.x) {
  const int lane = tid & 63, w = tid >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int ta = (w >> 1) & 1, tc = w & 1;
  const int kh = NW == 8 ? (w >> 2) : 0;
  const int ylo = NW == 8 ? kh * (N / 2) : 0;
  const int yhi = NW == 8 ? ylo + N / 2 : N;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // K steps of 32 in groups of 4 with the basis loads of a group in flight
  // together (the basis rows come from L2; one load per step would expose
  // its latency N/32 times)
  const int steps = (yhi - ylo) / 32;
  const bf16* xa = Xt + (long)(16 * ta + i) * ldx + ylo + 8 * g;
  const bf16* xb = lt + (16 * tc + i) * basis_ld(N) + ylo + 8 * g;
  for (int s0 = 0; s0 < steps; s0 += 4) {
    bf16x8 a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u < steps) a[u] = ld8(xa + 32 * (s0 + u));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u < steps) b[u] = ld8(xb + 32 * (s0 + u));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u < steps) acc = mma(a[u], b[u], acc);
  }
  if (NW == 8) {
    if (kh == 1) {
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((w & 3) * 64 + lane) * 4 + v] = acc[v];
    }
    __syncthreads();
    if (kh == 1) return;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] += red[(w * 64 + lane) * 4 + v];
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) o[(16 * ta + 4 * g + v) * C + 16 * tc + i] = acc[v];
}

// Input of the lift: sample k reads chi at k * sChi, v at k * sV and its
// norm at nrm + k * sNrm bytes (nrm null: v is used as it is).
struct LiftIn {
  const float* chi;
  long sChi;
  float chi_scale;
  const float2* v;
  long sV;
  const double* nrm;
  long sNrm;
  float s;          // v's scale (N: unit vectors become O(1) per cell)
  const float* P;   // W_in (3 x 32) followed by b_in (32)
};

// h0 of one cell at 8 channels c0..c0+7 from a = (chi chi_scale, s Re v',
// s Im v') and the lift parameters w (W_in rows 0-2 and b_in, channels
// c0..c0+7 at w[0..7], w[8..15], w[16..23], w[24..31]):
//   h0[c] = a0 W_in[0][c] + a1 W_in[1][c] + a2 W_in[2][c] + b_in[c]
// The one rounding of the lift: both row kernels that lift call this.
__device__ inline bf16x8 lift8(float a0, float a1, float a2, const float* w) {
  bf16x8 h;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    h[k] = (bf16)__builtin_fmaf(a2, w[16 + k], __builtin_fmaf(a1, w[8 + k], __builtin_fmaf(a0, w[k], w[24 + k])));
  return h;
}

// The lift of grid row xr of sample ks into the LDS row lt, channel-major
// [c][y] with row stride basis_ld(N) (TR) or [y][S], with (a0, a1, a2) =
// (chi chi_scale, s Re v', s Im v'), v' = v / *nrm: one item q = (cell y,
// quarter) of 8 channels per thread and step (the four items of a cell are
// adjacent lanes of one load, and a thread's loads all precede its stores,
// so an in-place vw == v is read before it is written).
// With h0 the row also goes to global memory (16-byte stores), with vw v'
// goes back to vw.  In two halves: lift_load issues the loads of one group
// of four items per thread (items q0 + u NT, clamped to the row, and the
// sample's norm, all unconditional), lift_store forms and stores them.
struct LiftRegs {
  float cv[4];
  float2 xv[4];
  double d;  // the sample's norm (1 without nrm)
};
template <int NT>
__device__ inline void lift_load(const LiftIn& L, long ks, int xr, int N, int q0, LiftRegs& g) {
  const long rin = (long)xr * N;  // the row's first cell in the sample
  const float* chi = L.chi + ks * L.sChi;
  const float2* v = L.v + ks * L.sV;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int q = q0 + u * NT < N * 4 ? q0 + u * NT : N * 4 - 1;
    g.cv[u] = chi[rin + (q >> 2)];
    g.xv[u] = v[rin + (q >> 2)];
  }
  // a global (not flat) load, which LDS waits do not wait for
  typedef __attribute__((address_space(1))) const double gdouble;
  g.d = *(gdouble*)(L.nrm ? boff(L.nrm, ks * L.sNrm) : &kOne);
}
// The 4 x 8 lift parameters of this thread's channels (NT % 4 == 0: every
// item of a thread has the same 8 channels).
__device__ inline void lift_weights(const LiftIn& L, float* w) {
  const int c8 = (threadIdx.x & 3) * 8;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
#pragma unroll
    for (int j = 0; j < 4; ++j) w[8 * j + k] = L.P[j * C + c8 + k];
  }
}
template <int NT, bool TR>
__device__ inline void lift_store(const LiftIn& L, const LiftRegs& g, const float* w, long ks, int xr, int N,
                                  int q0, bf16* lt, bf16* h0, float2* vw) {
  static_assert(NT % 4 == 0, "items of a thread must share their channels");
  const long rin = (long)xr * N;
  const int c8 = (threadIdx.x & 3) * 8;
  const float r = L.nrm ? (g.d > 0.0 ? (float)(1.0 / g.d) : 0.f) : 1.f;
  if (vw) vw += ks * L.sV;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int q = q0 + u * NT;
    if (q >= N * 4) break;
    const int y = q >> 2;
    const long pin = rin + y;
    float2 vv = g.xv[u];
    if (L.nrm) {
      vv.x *= r;
      vv.y *= r;
      if (vw && c8 == 0) vw[pin] = vv;
    }
    const bf16x8 hq = lift8(g.cv[u] * L.chi_scale, vv.x * L.s, vv.y * L.s, w);
    if (h0) *reinterpret_cast<u32x4*>(h0 + ((ks * N + xr) * N + y) * C + c8) = __builtin_bit_cast(u32x4, hq);
    if (TR) {
#pragma unroll
      for (int k = 0; k < 8; ++k) lt[(c8 + k) * basis_ld(N) + y] = hq[k];
    } else {
      const u32x4 bits = __builtin_bit_cast(u32x4, hq);
      u32x2* d = reinterpret_cast<u32x2*>(lt + y * S + c8);
      d[0] = u32x2{bits[0], bits[1]};
      d[1] = u32x2{bits[2], bits[3]};
    }
  }
}
template <int NT, bool TR>
__device__ inline void lift_row_to_lds(const LiftIn& L, long ks, int xr, int N, bf16* lt, bf16* h0,
                                       float2* vw) {
  float w[32];
  lift_weights(L, w);
  for (int q0 = threadIdx.x; q0 < N * 4; q0 += 4 * NT) {
    LiftRegs g;
    lift_load<NT>(L, ks, xr, N, q0, g);
    lift_store<NT, TR>(L, g, w, ks, xr, N, q0, lt, h0, vw);
  }
}

// One block (512 threads) per grid row x of one sample: the lift of the row
// to LDS (and to h0 when given: training keeps it for the backward pass),
// then its row projection into Aout[x].  With nrm the input is v / *nrm
// (written back to vw when given), which lets FGMRES hand over its lazily
// normalised Krylov vector.
__global__ void __launch_bounds__(512) k_lift_row(LiftIn L, float2* vw, bf16* __restrict__ h0,
                                                  const bf16* __restrict__ Xt, float* __restrict__ Aout, int N,
                                                  const int* done) {
  if (skip(done)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* lt = reinterpret_cast<bf16*>(smem_raw);  // the row, channel-major
  bf16* lbas = lt + C * basis_ld(N);
  __shared__ float red[4 * 64 * 4];
  const long bx = blockIdx.x;
  const long ks = bx / N;  // sample
  basis_to_lds<512>(Xt, lbas, N);
  lift_row_to_lds<512, true>(L, ks, (int)(bx - ks * N), N, lt, h0, vw);
  __syncthreads();
  row_project<8>(lbas, basis_ld(N), lt, N, Aout + bx * C * C, red);
}

// k_lift_row with RPW grid rows of one sample per block (N % RPW == 0 and
// N <= 512, one group of four items per thread): the basis is staged once,
// and each next row's chi and v are loaded before the current row's
// projection.
template <int RPW>
__global__ void __launch_bounds__(512) k_lift_rows(LiftIn L, float2* vw, bf16* __restrict__ h0,
                                                   const bf16* __restrict__ Xt, float* __restrict__ Aout, int N,
                                                   const int* done) {
  if (skip(done)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* lt = reinterpret_cast<bf16*>(smem_raw);  // the row, channel-major
  bf16* lbas = lt + C * basis_ld(N);
  __shared__ float red[4 * 64 * 4];
  const long bx0 = (long)blockIdx.x * RPW;
  const long ks = bx0 / N;  // sample of all RPW rows
  const int xr0 = (int)(bx0 - ks * N);
  LiftRegs g;
  lift_load<512>(L, ks, xr0, N, threadIdx.x, g);
  basis_to_lds<512>(Xt, lbas, N);
#pragma unroll
  for (int rr = 0; rr < RPW; ++rr) {
    if (rr) __syncthreads();  // the previous row's projection has read lt
    {
      float w[32];
      lift_weights(L, w);
      lift_store<512, true>(L, g, w, ks, xr0 + rr, N, threadIdx.x, lt, h0, vw);
    }
    __syncthreads();
    if (rr + 1 < RPW) lift_load<512>(L, ks, xr0 + rr + 1, N, threadIdx.x, g);
    row_project<8>(lbas, basis_ld(N), lt, N, Aout + (bx0 + rr) * C * C, red);
  }
}

// One block (8 waves) per grid row x of sample k (layers 0-2):
//   1. B_x to LDS (BF16), the MFMA A operand of the spectral half of the
//      GEMM: copied from R[k][x] (k_invx's output), or with FOLD formed
//      here as the inverse x-DFT of the mixed modes at this row (thread
//      (ky, o): B_x[o][2ky] + i B_x[o][2ky+1] = sum_kxi Vm[k][kxi][ky][o]
//      e^{+2 pi i kx x/N}), which saves k_invx's launch but reads all of
//      Vm[k] (128 KiB, from L2) per row: the better choice for one sample;
//   2. h'[y] = GELU([h[y], F_y] [W; B_x] + b) for the row's N cells (16-cell
//      tiles t = wave + 8u) to out (each lane stores the 4
//      channels it holds of one cell, 8 bytes) and channel-major into LDS
//      (pre-activations to pre_out when given, for training);
//   3. the row projection of h' into Anext[x], with the basis staged in LDS.
// With LIFT (layer 0) h[y] is not read from P: the row is lifted from (chi,
// v) into LDS as [y][S] first (lift_row_to_lds, the rounding of k_lift_row),
// 12 bytes per cell instead of 64, where the basis goes otherwise; the tiles
// read their cells from there, and the basis replaces the row after the
// tile loop.  (Lifting in registers per tile instead holds the 32 lift
// weights of a lane through the tile loop: 170 VGPRs, one work-group per CU;
// so does holding the basis in registers through the loop: 142 VGPRs.)
template <bool FOLD, bool LIFT>
__global__ void __launch_bounds__(512) k_cell_row(const bf16* __restrict__ P, LiftIn L, const bf16* __restrict__ Q,
                                                  const bf16* __restrict__ A, const bf16* __restrict__ R,
                                                  const float2* __restrict__ Vm, const float2* __restrict__ Ex,
                                                  const float* __restrict__ bias, bf16* __restrict__ pre_out,
                                                  bf16* __restrict__ out, const bf16* __restrict__ Xt,
                                                  float* __restrict__ Anext, int N, const int* done) {
  if (skip(done)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // region 1: the basis F^T (row stride basis_ld(N)); with LIFT first the
  // lifted row h0 as [y][S], the basis after the tiles have read it
  bf16* lbas = reinterpret_cast<bf16*>(smem_raw);
  bf16* lrow = lbas;
  bf16* lt = lbas + (N * S > C * basis_ld(N) ? N * S : C * basis_ld(N));  // region 2: h' channel-major
  __shared__ float red[4 * 64 * 4];
  __shared__ __align__(16) bf16 lb[C][C + 8];  // B_x as [o][k], rows padded to 80 B
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const long bx = blockIdx.x;  // sample * N + x
  const long ks = bx / N;
  const int xr = (int)(bx - ks * N);
  const int i = lane & 15, g = lane >> 4;
  const int ntile = N / 16;
  // the first tiles' cell operands and B_x are in flight while the basis
  // (or the lifted row) is staged; the loads are unconditional (tiles past
  // the row's end re-read its last tile, unused), so that no branch waits for
  // one load before the next is issued
  // the layer's weights and bias: loaded first, except with FOLD, whose
  // inverse x-DFT holds 64 registers of modes until B_x is formed
  bf16x8 aw[2];
  float bs[2][4];
  auto load_weights = [&]() {
#pragma unroll
    for (int to = 0; to < 2; ++to) {
      aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
#pragma unroll
      for (int v = 0; v < 4; ++v) bs[to][v] = bias[16 * to + 4 * g + v];
    }
  };
  if (!FOLD) load_weights();
  bf16x8 bpt[4], bqt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int t = w + 8 * u;
    t = t < ntile ? t : ntile - 1;
    const int y = 16 * t + i;
    if (!LIFT) bpt[u] = ld8(P + (bx * N + y) * C + 8 * g);
    bqt[u] = ld8(Q + (long)y * C + 8 * g);
  }
  u32x4 bxv;  // 128 threads x 8 BF16 of B_x (the other threads read a copy)
  if (!FOLD) bxv = *reinterpret_cast<const u32x4*>(R + (bx * C + ((tid >> 2) & 31)) * C + (tid & 3) * 8);
  if (LIFT)
    lift_row_to_lds<512, false>(L, ks, xr, N, lrow, nullptr, nullptr);
  else
    basis_to_lds<512>(Xt, lbas, N);
  if (!FOLD) {
    if (tid < C * C / 8) *reinterpret_cast<u32x4*>(&lb[tid >> 2][(tid & 3) * 8]) = bxv;
  } else {
    // the sums and their order of k_invx (rows x and N - x from the
    // twiddles of the pair's first row p), so one sample gets the B_x that
    // k_invx forms for a batch, bit for bit
    const int ky = tid >> 5, o = tid & 31;
    const float2* Vs = Vm + (ks * KX * KY + ky) * C + o;
    float2 vq[KX];
#pragma unroll
    for (int q = 0; q < KX; ++q) vq[q] = Vs[(long)q * KY * C];
    float bre, bim;
    if (xr == N / 2) {
      float t1 = 0.f, t2 = 0.f;
#pragma unroll
      for (int q = 0; q < KX; q += 2) {
        t1 += vq[q].x - vq[q + 1].x;
        t2 += vq[q].y - vq[q + 1].y;
      }
      bre = t1;
      bim = t2;
    } else {
      const int pr = xr < N / 2 ? xr : N - xr;
      float s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f;
#pragma unroll
      for (int q = 0; q < KX; ++q) {
        const float2 e = Ex[(long)q * N + pr];
        s1 += vq[q].x * e.x;
        s2 += vq[q].y * e.y;
        s3 += vq[q].x * e.y;
        s4 += vq[q].y * e.x;
      }
      bre = xr == pr ? s1 - s2 : s1 + s2;
      bim = xr == pr ? s3 + s4 : s4 - s3;
    }
    lb[o][2 * ky] = (bf16)bre;
    lb[o][2 * ky + 1] = (bf16)bim;
    load_weights();
  }
  __syncthreads();
  bf16x8 ar[2];
#pragma unroll
  for (int to = 0; to < 2; ++to) ar[to] = *reinterpret_cast<const bf16x8*>(&lb[16 * to + i][8 * g]);
  // LIFT with at most four tiles per wave (N <= 512): every wave takes its
  // cells from the lifted row first, then the basis replaces the row before
  // the tile loop, its load latency hidden by the other waves' GEMMs
  // (block-uniform branch)
  const bool early = LIFT && ntile <= 32;
  if (early) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      int t = w + 8 * u;
      t = t < ntile ? t : ntile - 1;
      const u32x2* sp = reinterpret_cast<const u32x2*>(lrow + (16 * t + i) * S + 8 * g);
      const u32x2 lo = sp[0], hi = sp[1];
      bpt[u] = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
    __syncthreads();
    basis_to_lds<512>(Xt, lbas, N);
  }
  for (int k0 = 0; w + 8 * k0 < ntile; k0 += 4) {
    if (k0 > 0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int t = w + 8 * (k0 + u);
        t = t < ntile ? t : ntile - 1;
        const int y = 16 * t + i;
        if (!LIFT) bpt[u] = ld8(P + (bx * N + y) * C + 8 * g);
        bqt[u] = ld8(Q + (long)y * C + 8 * g);
      }
    }
    if (LIFT && !early) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = w + 8 * (k0 + u);
        if (t < ntile) {
          const u32x2* sp = reinterpret_cast<const u32x2*>(lrow + (16 * t + i) * S + 8 * g);
          const u32x2 lo = sp[0], hi = sp[1];
          bpt[u] = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = w + 8 * (k0 + u);
      if (t >= ntile) break;
      const int y = 16 * t + i;
#pragma unroll
      for (int to = 0; to < 2; ++to) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mma(aw[to], bpt[u], acc);
        acc = mma(ar[to], bqt[u], acc);
        const int oc0 = 16 * to + 4 * g;
        float r[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = acc[v] + bs[to][v];
        if (pre_out) st4(pre_out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = gelu(r[v]);
        st4(out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) lt[(oc0 + v) * basis_ld(N) + y] = (bf16)r[v];
      }
    }
  }
  __syncthreads();
  if (LIFT && !early) {  // the lifted row is dead: the basis takes its place
    basis_to_lds<512>(Xt, lbas, N);
    __syncthreads();
  }
  row_project<8>(lbas, basis_ld(N), lt, N, Anext + bx * C * C, red);
}

// k_cell_row<true, LIFT> on the two grid rows of a pair (p, N - p; 0 and N/2
// for p = 0) of one sample, 512 threads per row, for N <= 512 (a wave owns at
// most four 16-cell tiles; both rows fit the LDS).  The pair's B_x come from
// the same four sums, so the modes are read and summed once for two rows, and
// the basis is staged once.  The arithmetic of a row is k_cell_row's.  At
// N = 512: 14.4 us (lifting 15.3), where single rows, two work-groups per CU,
// take 16.4 (16.7), 3 of them for the modes.
inline size_t cell_pair_lds(int N, bool lift) {
  const size_t t = (size_t)C * basis_ld(N), r = (size_t)2 * N * S;
  return (2 * t + (lift && r > t ? r : t)) * sizeof(bf16);
}
template <bool LIFT>
__global__ void __launch_bounds__(1024) k_cell_pair(const bf16* __restrict__ P, LiftIn L,
                                                    const bf16* __restrict__ Q, const bf16* __restrict__ A,
                                                    const float2* __restrict__ Vm, const float2* __restrict__ Ex,
                                                    const float* __restrict__ bias, bf16* __restrict__ pre_out,
                                                    bf16* __restrict__ out, const bf16* __restrict__ Xt,
                                                    float* __restrict__ Anext, int N, const int* done) {
  if (skip(done)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ float red[2][4 * 64 * 4];
  __shared__ __align__(16) bf16 lb[2][C][C + 8];  // B_x of the two rows as [o][k], rows padded to 80 B
  const int half = threadIdx.x >> 9, tid = threadIdx.x & 511, lane = tid & 63, w = tid >> 6;
  const int p = blockIdx.x;  // the pair's first row
  const int xr = half == 0 ? p : p == 0 ? N / 2 : N - p;
  const long ks = blockIdx.y, bx = ks * N + xr;
  bf16* lt = reinterpret_cast<bf16*>(smem_raw) + half * C * basis_ld(N);  // h' channel-major
  bf16* lbas = reinterpret_cast<bf16*>(smem_raw) + 2 * C * basis_ld(N);   // the basis, with LIFT first
  bf16* lrow = lbas + half * N * S;                                       // the lifted rows
  const int i = lane & 15, g = lane >> 4;
  const int ntile = N / 16;
  bf16x8 bpt[4], bqt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int t = w + 8 * u;
    t = t < ntile ? t : ntile - 1;
    const int y = 16 * t + i;
    if (!LIFT) bpt[u] = ld8(P + (bx * N + y) * C + 8 * g);
    bqt[u] = ld8(Q + (long)y * C + 8 * g);
  }
  if (LIFT) {
    float wl[32];
    lift_weights(L, wl);
    for (int q0 = tid; q0 < N * 4; q0 += 4 * 512) {
      LiftRegs lg;
      lift_load<512>(L, ks, xr, N, q0, lg);
      lift_store<512, false>(L, lg, wl, ks, xr, N, q0, lrow, nullptr, nullptr);
    }
  }
  if (half == 0) {  // the sums and their order of k_invx
    const int ky = tid >> 5, o = tid & 31;
    const float2* Vs = Vm + (ks * KX * KY + ky) * C + o;
    float2 vq[KX];
#pragma unroll
    for (int q = 0; q < KX; ++q) vq[q] = Vs[(long)q * KY * C];
    float s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f;
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const float2 e = Ex[(long)q * N + p];
      s1 += vq[q].x * e.x;
      s2 += vq[q].y * e.y;
      s3 += vq[q].x * e.y;
      s4 += vq[q].y * e.x;
    }
    lb[0][o][2 * ky] = (bf16)(s1 - s2);
    lb[0][o][2 * ky + 1] = (bf16)(s3 + s4);
    if (p == 0) {  // row N/2
      s1 = s4 = s2 = s3 = 0.f;
#pragma unroll
      for (int q = 0; q < KX; q += 2) {
        s1 += vq[q].x - vq[q + 1].x;
        s4 += vq[q].y - vq[q + 1].y;
      }
    }
    lb[1][o][2 * ky] = (bf16)(s1 + s2);
    lb[1][o][2 * ky + 1] = (bf16)(s4 - s3);
  } else if (!LIFT) {
    basis_to_lds<512>(Xt, lbas, N, tid);
  }
  bf16x8 aw[2];
  float bs[2][4];
#pragma unroll
  for (int to = 0; to < 2; ++to) {
    aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
#pragma unroll
    for (int v = 0; v < 4; ++v) bs[to][v] = bias[16 * to + 4 * g + v];
  }
  __syncthreads();
  bf16x8 ar[2];
#pragma unroll
  for (int to = 0; to < 2; ++to) ar[to] = *reinterpret_cast<const bf16x8*>(&lb[half][16 * to + i][8 * g]);
  if (LIFT) {  // every wave takes its cells, then the basis replaces the rows
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      int t = w + 8 * u;
      t = t < ntile ? t : ntile - 1;
      const u32x2* sp = reinterpret_cast<const u32x2*>(lrow + (16 * t + i) * S + 8 * g);
      const u32x2 lo = sp[0], hi = sp[1];
      bpt[u] = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
    __syncthreads();
    basis_to_lds<1024>(Xt, lbas, N);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int t = w + 8 * u;
    if (t >= ntile) break;
    const int y = 16 * t + i;
#pragma unroll
    for (int to = 0; to < 2; ++to) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = mma(aw[to], bpt[u], acc);
      acc = mma(ar[to], bqt[u], acc);
      const int oc0 = 16 * to + 4 * g;
      float r[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = acc[v] + bs[to][v];
      if (pre_out) st4(pre_out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = gelu(r[v]);
      st4(out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
      for (int v = 0; v < 4; ++v) lt[(oc0 + v) * basis_ld(N) + y] = (bf16)r[v];
    }
  }
  __syncthreads();
  row_project<8>(lbas, basis_ld(N), lt, N, Anext + bx * C * C, red[half], tid);
}

// k_cell_row<false, false> (B_x from R, the cells from P) with RPW
// consecutive rows per work-group, for N <= 512 (a wave owns at most four
// 16-cell tiles, the same ones in every row).  The basis F^T, the layer's
// weights and the F_y operands are staged once for the RPW rows, and the
// next row's cells and B_x are loaded before the current row's projection,
// so that the HBM reads of one row overlap the LDS work of the other.  The
// arithmetic of a row is k_cell_row's, operation for operation.
template <int RPW>
__global__ void __launch_bounds__(512) k_cell_rows(const bf16* __restrict__ P, const bf16* __restrict__ Q,
                                                   const bf16* __restrict__ A, const bf16* __restrict__ R,
                                                   const float* __restrict__ bias, bf16* __restrict__ pre_out,
                                                   bf16* __restrict__ out, const bf16* __restrict__ Xt,
                                                   float* __restrict__ Anext, int N, const int* done) {
  if (skip(done)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* lbas = reinterpret_cast<bf16*>(smem_raw);  // the basis F^T
  bf16* lt = lbas + C * basis_ld(N);               // h' of the row, channel-major
  __shared__ float red[4 * 64 * 4];
  __shared__ __align__(16) bf16 lb[C][C + 8];  // B_x as [o][k]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int ntile = N / 16;
  const long bx0 = (long)blockIdx.x * RPW;  // sample * N + x of the first row
  bf16x8 aw[2];
  float bs[2][4];
#pragma unroll
  for (int to = 0; to < 2; ++to) {
    aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
#pragma unroll
    for (int v = 0; v < 4; ++v) bs[to][v] = bias[16 * to + 4 * g + v];
  }
  bf16x8 bpt[4], bqt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int t = w + 8 * u;
    t = t < ntile ? t : ntile - 1;
    const int y = 16 * t + i;
    bpt[u] = ld8(P + (bx0 * N + y) * C + 8 * g);
    bqt[u] = ld8(Q + (long)y * C + 8 * g);
  }
  const int bxo = (((tid >> 2) & 31)) * C + (tid & 3) * 8;  // this thread's 8 BF16 of B_x
  u32x4 bxv = *reinterpret_cast<const u32x4*>(R + bx0 * C * C + bxo);
  basis_to_lds<512>(Xt, lbas, N);
  // unrolled: as a loop the row-invariant addresses stay live across the
  // iterations (about 155 VGPRs, one work-group per CU); unrolled it needs
  // 109 at RPW 2 and 121 at RPW 4 and 8, two work-groups per CU
#pragma unroll
  for (int rr = 0; rr < RPW; ++rr) {
    const long bx = bx0 + rr;
    if (tid < C * C / 8) *reinterpret_cast<u32x4*>(&lb[tid >> 2][(tid & 3) * 8]) = bxv;
    __syncthreads();
    bf16x8 ar[2];
#pragma unroll
    for (int to = 0; to < 2; ++to) ar[to] = *reinterpret_cast<const bf16x8*>(&lb[16 * to + i][8 * g]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = w + 8 * u;
      if (t >= ntile) break;
      const int y = 16 * t + i;
#pragma unroll
      for (int to = 0; to < 2; ++to) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mma(aw[to], bpt[u], acc);
        acc = mma(ar[to], bqt[u], acc);
        const int oc0 = 16 * to + 4 * g;
        float r[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = acc[v] + bs[to][v];
        if (pre_out) st4(pre_out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = gelu(r[v]);
        st4(out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) lt[(oc0 + v) * basis_ld(N) + y] = (bf16)r[v];
      }
    }
    __syncthreads();
    if (rr + 1 < RPW) {  // the next row's operands (block-uniform branch)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int t = w + 8 * u;
        t = t < ntile ? t : ntile - 1;
        bpt[u] = ld8(P + ((bx + 1) * N + 16 * t + i) * C + 8 * g);
      }
      bxv = *reinterpret_cast<const u32x4*>(R + (bx + 1) * C * C + bxo);
    }
    // waves of the upper K half leave row_project after its barrier; every
    // wave has read lt and red of this row before the next row's first
    // barrier, after which they are written again
    row_project<8>(lbas, basis_ld(N), lt, N, Anext + bx * C * C, red);
  }
}

// k_cell_row<false, true> (layer 0 of a batch) with RPW grid rows of one
// sample per block, N % RPW == 0 and N <= 512.  One LDS region holds the
// basis for all rows; the other holds a row lifted from (chi, v) as [y][S]
// until every wave has taken its cells, then h' channel-major for the row
// projection.  The weights, the F_y operands and the basis are loaded once;
// each next row's chi, v and B_x are loaded before the current row's
// projection.  The arithmetic of a row is k_cell_row's.
template <int RPW>
__global__ void __launch_bounds__(512) k_cell_rows_lift(LiftIn L, const bf16* __restrict__ Q,
                                                         const bf16* __restrict__ A, const bf16* __restrict__ R,
                                                         const float* __restrict__ bias, bf16* __restrict__ pre_out,
                                                         bf16* __restrict__ out, const bf16* __restrict__ Xt,
                                                         float* __restrict__ Anext, int N, const int* done) {
  if (skip(done)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* lbas = reinterpret_cast<bf16*>(smem_raw);  // the basis F^T
  bf16* lx = lbas + C * basis_ld(N);               // the lifted row, then h'
  __shared__ float red[4 * 64 * 4];
  __shared__ __align__(16) bf16 lb[C][C + 8];  // B_x as [o][k]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int ntile = N / 16;
  const long bx0 = (long)blockIdx.x * RPW;
  const long ks = bx0 / N;  // sample of all RPW rows
  const int xr0 = (int)(bx0 - ks * N);
  bf16x8 aw[2];
  float bs[2][4];
#pragma unroll
  for (int to = 0; to < 2; ++to) {
    aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
#pragma unroll
    for (int v = 0; v < 4; ++v) bs[to][v] = bias[16 * to + 4 * g + v];
  }
  bf16x8 bqt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int t = w + 8 * u;
    t = t < ntile ? t : ntile - 1;
    bqt[u] = ld8(Q + (long)(16 * t + i) * C + 8 * g);
  }
  const int bxo = ((tid >> 2) & 31) * C + (tid & 3) * 8;  // this thread's 8 BF16 of B_x
  u32x4 bxv = *reinterpret_cast<const u32x4*>(R + bx0 * C * C + bxo);
  LiftRegs lg;
  lift_load<512>(L, ks, xr0, N, tid, lg);
  basis_to_lds<512>(Xt, lbas, N);
#pragma unroll
  for (int rr = 0; rr < RPW; ++rr) {
    const long bx = bx0 + rr;
    if (rr) __syncthreads();  // the previous row's projection has read lx
    {
      float wl[32];
      lift_weights(L, wl);
      lift_store<512, false>(L, lg, wl, ks, xr0 + rr, N, tid, lx, nullptr, nullptr);
    }
    if (tid < C * C / 8) *reinterpret_cast<u32x4*>(&lb[tid >> 2][(tid & 3) * 8]) = bxv;
    __syncthreads();
    bf16x8 ar[2], bpt[4];
#pragma unroll
    for (int to = 0; to < 2; ++to) ar[to] = *reinterpret_cast<const bf16x8*>(&lb[16 * to + i][8 * g]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      int t = w + 8 * u;
      t = t < ntile ? t : ntile - 1;
      const u32x2* sp = reinterpret_cast<const u32x2*>(lx + (16 * t + i) * S + 8 * g);
      const u32x2 lo = sp[0], hi = sp[1];
      bpt[u] = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
    __syncthreads();  // every wave has its cells: lx takes h'
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = w + 8 * u;
      if (t >= ntile) break;
      const int y = 16 * t + i;
#pragma unroll
      for (int to = 0; to < 2; ++to) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mma(aw[to], bpt[u], acc);
        acc = mma(ar[to], bqt[u], acc);
        const int oc0 = 16 * to + 4 * g;
        float r[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = acc[v] + bs[to][v];
        if (pre_out) st4(pre_out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = gelu(r[v]);
        st4(out + (bx * N + y) * C + oc0, r[0], r[1], r[2], r[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) lx[(oc0 + v) * basis_ld(N) + y] = (bf16)r[v];
      }
    }
    __syncthreads();
    if (rr + 1 < RPW) {  // the next row's operands
      lift_load<512>(L, ks, xr0 + rr + 1, N, tid, lg);
      bxv = *reinterpret_cast<const u32x4*>(R + (bx + 1) * C * C + bxo);
    }
    row_project<8>(lbas, basis_ld(N), lx, N, Anext + bx * C * C, red);
  }
}

// Layer 3 (no activation) fused with the projection: per cell
//   h4 = [h3, F_y] [W; B_x] + b,  z = s_id vv / *vnrm + (h4 W_out + b_out) / s
// in FP32 (vnrm null: no scaling); h4 goes to hout as BF16 when given
// (training).  Sample k reads vv and writes z at k * sV, k * sZ, its norm at
// vnrm + k * sNrm bytes.  One wave per 64 cells, as k_back_cells.
__global__ void __launch_bounds__(256) k_cell_proj(const bf16* __restrict__ P, const bf16* __restrict__ Q,
                                                   const bf16* __restrict__ A, const bf16* __restrict__ R,
                                                   const float* __restrict__ bias, bf16* __restrict__ hout,
                                                   const float* __restrict__ Pp, const float2* __restrict__ vv,
                                                   long sV, const double* vnrm, long sNrm, float s,
                                                   float2* __restrict__ z, long sZ, int N, const int* done) {
  if (skip(done)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const long wv = (long)blockIdx.x * 4 + w;  // every block is full: waves % 4 == 0
  const int segs = N / 64;
  const long bx = wv / segs;
  const int y0 = (int)(wv % segs) * 64;
  const int i = lane & 15, g = lane >> 4;
  const long ks = bx / N;                 // sample
  const long rin = (bx - ks * N) * N;     // the row's first cell in the sample
  vv += ks * sV;
  z += ks * sZ;
  // every load of the wave is issued before the first use of any: the cell
  // operands, the vector's values, the weights, then the vector's norm (read
  // through a pointer that is never null, so that no branch waits for the
  // loads before it)
  bf16x8 bpt[4], bqt[4];
  float2 vx[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int y = y0 + 16 * t + i;
    bpt[t] = ld8(P + (bx * N + y) * C + 8 * g);
    bqt[t] = ld8(Q + (long)y * C + 8 * g);
    vx[t] = vv[rin + y];
  }
  bf16x8 aw[2], ar[2];
  float bs[2][4], wo[2][4][2];
  const float* Wout = Pp + kOffOut;
#pragma unroll
  for (int to = 0; to < 2; ++to) {
    aw[to] = ld8(A + (16 * to + i) * C + 8 * g);
    ar[to] = ld8(R + (bx * C + 16 * to + i) * C + 8 * g);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int o = 16 * to + 4 * g + v;
      bs[to][v] = bias[o];
      wo[to][v][0] = Wout[2 * o];
      wo[to][v][1] = Wout[2 * o + 1];
    }
  }
  const double d = *(vnrm ? boff(vnrm, ks * sNrm) : &kOne);  // no norm: 1
  const float sid = Pp[kOffSkip] * (d > 0.0 ? (float)(1.0 / d) : 0.f);
  const float b0 = Wout[2 * C], b1 = Wout[2 * C + 1], is = 1.f / s;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const long p = bx * N + y0 + 16 * t + i;
    float o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int to = 0; to < 2; ++to) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = mma(aw[to], bpt[t], acc);
      acc = mma(ar[to], bqt[t], acc);
      float r[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        r[v] = acc[v] + bs[to][v];
        o0 += r[v] * wo[to][v][0];
        o1 += r[v] * wo[to][v][1];
      }
      if (hout) st4(hout + p * C + 16 * to + 4 * g, r[0], r[1], r[2], r[3]);
    }
    // the four lane groups g hold channels 4g..4g+3 (+16) of cell i
    o0 += __shfl_xor(o0, 16, 64);
    o1 += __shfl_xor(o1, 16, 64);
    o0 += __shfl_xor(o0, 32, 64);
    o1 += __shfl_xor(o1, 32, 64);
    if (g == 0) {
      const float2 x = vx[t];
      z[rin + y0 + 16 * t + i] = make_float2(sid * x.x + (o0 + b0) * is, sid * x.y + (o1 + b1) * is);
    }
  }
}


// Gradients of the projection and of the identity path, with d = dz / s:
//   part[blk] = (sum_p h[p][c] d_j  [c][j],  sum_p d_j,  sum_p Re(conj(dz) v))
// Bound by the read of h, 64 bytes per cell: four lanes share a cell, 8
// channels each, so a wave reads 1 KiB at once: 12 us at N = 256, 8 samples
// (512 blocks 17; with one lane per cell and dh4 stored 26).
__global__ void __launch_bounds__(256) k_proj_bwd(const float2* __restrict__ dz, const bf16* __restrict__ h,
                                                  const float2* __restrict__ v, float is,
                                                  float* __restrict__ part, long total) {
  __shared__ float red[4][2 * C + 3];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c8 = (tid & 3) * 8;
  float acc[16] = {}, s0 = 0.f, s1 = 0.f, s2 = 0.f;
  constexpr int U = 4;  // cells per thread and step, in flight together
  const long step = (long)gridDim.x * 64;
  for (long p0 = (long)blockIdx.x * 64 + (tid >> 2); p0 < total; p0 += U * step) {
    bf16x8 hv[U];
    float2 d[U], vv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long p = p0 + u * step < total ? p0 + u * step : total - 1;
      hv[u] = ld8(h + p * C + c8);
      d[u] = dz[p];
      vv[u] = v[p];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (p0 + u * step >= total) break;
      const float d0 = d[u].x * is, d1 = d[u].y * is;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float x = (float)hv[u][k];
        acc[2 * k] += x * d0;
        acc[2 * k + 1] += x * d1;
      }
      s0 += d0;
      s1 += d1;
      s2 += d[u].x * vv[u].x + d[u].y * vv[u].y;
    }
  }
  auto join = [&](float t) {
#pragma unroll
    for (int m = 4; m < 64; m *= 2) t += __shfl_xor(t, m, 64);
    return t;
  };
  lane16_sums<16, 4>(acc, lane >> 2);
  red[w][2 * c8 + (lane >> 2)] = acc[0];
  s0 = join(s0);
  s1 = join(s1);
  s2 = join(s2);
  if (lane == 0) {
    red[w][2 * C] = s0;
    red[w][2 * C + 1] = s1;
    red[w][2 * C + 2] = s2;
  }
  __syncthreads();
  if (tid < 2 * C + 3)
    part[(long)blockIdx.x * (2 * C + 3) + tid] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
}

// out[k] = sum_g part[g * width + k] for every segment of the backward pass
// (projection, the layers' weights and biases, lift) in one launch: 64 outputs per
// block, 16 strided slices of g per output combined in a fixed order, sixteen
// loads of a slice in flight: 8 us, where a launch per reduction took 6 x 6.
struct ReduceSeg {
  const float* part;
  float* out;
  int G, width, block0;  // block0: the segment's first block
};
constexpr int kReduceSegs = 6;
struct ReduceList {
  ReduceSeg seg[kReduceSegs];
};
__global__ void __launch_bounds__(1024) k_reduce_part(ReduceList list) {
  __shared__ float red[16][65];
  ReduceSeg q = list.seg[0];
#pragma unroll
  for (int j = 1; j < kReduceSegs; ++j)
    if ((int)blockIdx.x >= list.seg[j].block0) q = list.seg[j];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int k = (blockIdx.x - q.block0) * 64 + tx;
  float s = 0.f;
  if (k < q.width)
    for (int g0 = ty; g0 < q.G; g0 += 256) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int gi = g0 + 16 * u;
        v[u] = q.part[(long)(gi < q.G ? gi : ty) * q.width + k];
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) s += g0 + 16 * u < q.G ? v[u] : 0.f;
    }
  red[ty][tx] = s;
  __syncthreads();
  if (ty == 0 && k < q.width) {
    float t = 0.f;
    for (int e = 0; e < 16; ++e) t += red[e][tx];
    q.out[k] = t;
  }
}

// GEMM weights to BF16: Wt[l][o][c] = W_l[c][o] (forward A operand),
// Wn[l][c][o] = W_l[c][o] (backward A operand).
__global__ void __launch_bounds__(256) k_prep(const float* __restrict__ P, bf16* __restrict__ Wt,
                                              bf16* __restrict__ Wn) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= 4 * C * C) return;
  const int l = e / (C * C), r = e % (C * C), c = r / C, o = r % C;
  const float w = P[layer_off(l) + r];
  Wn[e] = (bf16)w;
  Wt[l * C * C + o * C + c] = (bf16)w;
}

}  // namespace fno
}  // namespace cgm

using namespace cgm;
using namespace cgm::fno;

struct cgm_fno {
  cgm_context* ctx = nullptr;
  int device = 0;  // kept here so the network can be destroyed after its context
  int N = 0, B = 0;
  long n = 0;
  float chi_scale = 1.f;
  const float* params = nullptr;  // caller's FP32 parameters (device)
  bf16* Wt = nullptr;             // 4 x 32 x 32
  bf16* Wn = nullptr;
  bf16* Ft = nullptr;             // 32 x N
  bf16* Fy = nullptr;             // N x 32
  float2* Ex = nullptr;           // [32 kxi][N]: e^{2 pi i kx x/N}
  bf16* h[5] = {};                // activations [B][n][32]
  bf16* pre[3] = {};              // pre-activations (training)
  bf16* dh[2] = {};               // backward ping-pong
  float* A = nullptr;             // [B][N][32][32]
  float2* U[4] = {};              // [B][32][16][32] (training)
  float2* dV[4] = {};             // [B][32][16][32] per layer
  float2* Vm = nullptr;           // [B][32][16][32] mixed modes
  bf16* Bt = nullptr;             // [B][N][32][32]
  float* part = nullptr;          // reduction partials
  // saved by the last training forward
  int fwd_batch = 0;
  const float* chi_in = nullptr;
  const float2* v_in = nullptr;
};

namespace {

int fno_free(cgm_fno* f) {
  void* ptrs[] = {f->Wt, f->Wn, f->Ft, f->Fy, f->Ex, f->h[0], f->h[1], f->h[2], f->h[3], f->h[4],
                  f->pre[0], f->pre[1], f->pre[2], f->dh[0], f->dh[1], f->A, f->U[0],
                  f->U[1], f->U[2], f->U[3], f->dV[0], f->dV[1], f->dV[2], f->dV[3], f->Vm, f->Bt, f->part};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  return CGM_SUCCESS;
}

// Blocks of the backward pass's reducing kernels: two row kernels per CU
// (each holds the next row's loads in flight), enough waves of the two cell
// kernels to fill the chip; each block leaves one set of partials.
int back_rows_grid(int rows) { return rows < 512 ? rows : 512; }
int back_cells_grid(long nseg) { return nseg / 4 < 1024 ? (int)(nseg / 4) : 1024; }
constexpr int kProjGrid = 1024;
constexpr int kRowPart = C * C + C, kProjPart = 2 * C + 3, kLiftPart = 4 * C;

// k_back_rows of a layer: Y, or dz with the output weights when Y is null.
template <int NC>
void launch_back_rows_n(const cgm_fno* f, hipStream_t st, const bf16* Y, const float2* dz, const bf16* Z,
                        float* part, int B) {
  const int rows = B * f->N;
  const size_t lds = (size_t)2 * f->N * C * sizeof(bf16);
  const float* Wout = f->params + kOffOut;
  const float is = 1.f / (float)f->N;
  const dim3 grid(back_rows_grid(rows)), block(512);
  if (Y)
    hipLaunchKernelGGL((k_back_rows<NC, false>), grid, block, lds, st, f->Ft, Y, dz, Wout, is, Z, f->A, part,
                       f->N, rows);
  else
    hipLaunchKernelGGL((k_back_rows<NC, true>), grid, block, lds, st, f->Ft, Y, dz, Wout, is, Z, f->A, part,
                       f->N, rows);
}
int launch_back_rows(const cgm_fno* f, hipStream_t st, const bf16* Y, const float2* dz, const bf16* Z, float* part,
                     int B) {
  if (f->N <= 128)
    launch_back_rows_n<1>(f, st, Y, dz, Z, part, B);
  else if (f->N <= 256)
    launch_back_rows_n<2>(f, st, Y, dz, Z, part, B);
  else if (f->N <= 512)
    launch_back_rows_n<4>(f, st, Y, dz, Z, part, B);
  else
    launch_back_rows_n<8>(f, st, Y, dz, Z, part, B);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

// One row pair per work-group while that is at most one per CU, then two, four
// from twice as many on, and eight where they still give every CU one: the
// forward pass of three samples of N = 320 (480 pairs) takes 124.5 us with two
// and 130.1 with one, of two of N = 256 (256 pairs) 86.2 and 85.1; eight samples
// of N = 256 (1,024 pairs): k_invx 7.0 us with four, 8.9 with eight.
void launch_invx(cgm_fno* f, hipStream_t st, int B, const int* done) {
  const int pairs = f->N / 2 * B;
  if (pairs >= 8 * 256)
    hipLaunchKernelGGL(k_invx<8>, dim3(f->N / 16, 1, B), dim3(512), 0, st, f->Vm, f->Bt, f->Ex, f->N, done);
  else if (pairs > 2 * 256)
    hipLaunchKernelGGL(k_invx<4>, dim3(f->N / 8, 1, B), dim3(512), 0, st, f->Vm, f->Bt, f->Ex, f->N, done);
  else if (pairs > 256)
    hipLaunchKernelGGL(k_invx<2>, dim3(f->N / 4, 1, B), dim3(512), 0, st, f->Vm, f->Bt, f->Ex, f->N, done);
  else
    hipLaunchKernelGGL(k_invx<1>, dim3(f->N / 2, 1, B), dim3(512), 0, st, f->Vm, f->Bt, f->Ex, f->N, done);
}

// A of B vectors to the mixed modes Vm, with the fewest frequencies per block
// (2, 4, 8, 16) that need no more than 256 blocks: the LDS holds one block per
// CU, so more of them are a second round (8 samples of N = 256: 16 per block
// 11.4 us, 8 per block 15.9; one of N = 512: 2 per block 7.9, 4 per block 8.7;
// six of N = 512: 8 per block 20.8, 16 per block 13.5).
template <int KG, bool SIX>
void launch_spectral_k(const cgm_fno* f, hipStream_t st, const float2* W, float2* usave, bool bwd, int B,
                       const int* done) {
  typedef SpecShape<KG, SIX> Sh;
  hipLaunchKernelGGL((bwd ? k_spectral<KG, true, SIX> : k_spectral<KG, false, SIX>), dim3(KY, KX / KG, B),
                     dim3(Sh::NTHR), Sh::lds(f->N), st, f->A, f->Ex, W, usave, f->Vm, f->N, done);
}
template <int KG>
void launch_spectral_n(const cgm_fno* f, hipStream_t st, const float2* W, float2* usave, bool bwd, int B,
                       const int* done) {
  const int nch = f->N / 64;
  if constexpr (KG >= 8) {
    if (nch == 5 || nch == 6) return launch_spectral_k<KG, true>(f, st, W, usave, bwd, B, done);
  }
  launch_spectral_k<KG, false>(f, st, W, usave, bwd, B, done);
}
void launch_spectral(const cgm_fno* f, hipStream_t st, const float2* W, float2* usave, bool bwd, int B,
                     const int* done) {
  const int kg = KY * KX * B / 256;  // at least this many
  if (kg > 8)
    launch_spectral_n<16>(f, st, W, usave, bwd, B, done);
  else if (kg > 4)
    launch_spectral_n<8>(f, st, W, usave, bwd, B, done);
  else if (kg > 2)
    launch_spectral_n<4>(f, st, W, usave, bwd, B, done);
  else
    launch_spectral_n<2>(f, st, W, usave, bwd, B, done);
}
// Lets a kernel ask for all the LDS that its static part leaves.  The limit
// belongs to the kernel, not to a network: one set to what this network's N
// needs would be lowered by a smaller network created later.
int whole_lds(const void* kernel) {
  hipFuncAttributes at;
  CGM_HIP(hipFuncGetAttributes(&at, kernel));
  CGM_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)(kMaxLds - at.sharedSizeBytes)));
  return CGM_SUCCESS;
}
template <int KG, bool SIX>
constexpr const void* spectral_kernel(bool bwd) {
  return bwd ? (const void*)k_spectral<KG, true, SIX> : (const void*)k_spectral<KG, false, SIX>;
}
// Of every kernel with an N-dependent LDS size, on the current device.
int lds_limits() {
  const void* kernels[] = {
      spectral_kernel<2, false>(false),       spectral_kernel<2, false>(true),
      spectral_kernel<4, false>(false),       spectral_kernel<4, false>(true),
      spectral_kernel<8, false>(false),       spectral_kernel<8, false>(true),
      spectral_kernel<16, false>(false),      spectral_kernel<16, false>(true),
      spectral_kernel<8, true>(false),        spectral_kernel<8, true>(true),
      spectral_kernel<16, true>(false),       spectral_kernel<16, true>(true),
      (const void*)k_back_rows<1, false>,     (const void*)k_back_rows<1, true>,
      (const void*)k_back_rows<2, false>,     (const void*)k_back_rows<2, true>,
      (const void*)k_back_rows<4, false>,     (const void*)k_back_rows<4, true>,
      (const void*)k_back_rows<8, false>,     (const void*)k_back_rows<8, true>,
      (const void*)k_lift_row,                (const void*)k_cell_pair<false>,
      (const void*)k_cell_pair<true>,         (const void*)k_cell_row<true, false>,
      (const void*)k_cell_row<false, false>,  (const void*)k_cell_row<true, true>,
      (const void*)k_cell_row<false, true>,   (const void*)k_cell_rows<2>,
      (const void*)k_cell_rows<4>,            (const void*)k_cell_rows<8>,
      (const void*)k_cell_rows_lift<2>,       (const void*)k_cell_rows_lift<4>,
      (const void*)k_lift_rows<2>,            (const void*)k_lift_rows<4>};
  for (const void* k : kernels) {
    const int rc = whole_lds(k);
    if (rc) return rc;
  }
  return CGM_SUCCESS;
}

// spectral path of one layer: A (row projections) -> Bt (per-row mixing matrices)
int spectral(cgm_fno* f, hipStream_t st, const float2* W, float2* usave, bool bwd, int B, const int* done,
             bool invx = true) {
  launch_spectral(f, st, W, usave, bwd, B, done);
  if (invx)
    launch_invx(f, st, B, done);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

}  // namespace

namespace cgm {

// Two grid rows per block where N allows it (N even, N <= 512) and the
// grid still holds at least 512 blocks, two per CU, from as many on four: one pass
// over four samples of N = 256 takes 106 us (116.6 with single rows), over four of
// N = 512 211 with four rows per block and 221 with two.
inline bool two_rows(int N, int rows) { return N % 2 == 0 && N <= 512 && rows / 2 >= 512; }

// The lift with layer 0's first row projection (k_lift_row / k_lift_rows):
// four rows per block where the grid still holds 512 blocks, else two.
void launch_lift(const cgm_fno* f, hipStream_t st, int rows, const LiftIn& L, float2* vw, bf16* h0,
                 const int* done) {
  const size_t lds = row_kernel_lds(f->N);
  if (f->N % 4 == 0 && f->N <= 512 && rows / 4 >= 512)
    hipLaunchKernelGGL(k_lift_rows<4>, dim3(rows / 4), dim3(512), lds, st, L, vw, h0, f->Ft, f->A, f->N, done);
  else if (two_rows(f->N, rows))
    hipLaunchKernelGGL(k_lift_rows<2>, dim3(rows / 2), dim3(512), lds, st, L, vw, h0, f->Ft, f->A, f->N, done);
  else
    hipLaunchKernelGGL(k_lift_row, dim3(rows), dim3(512), lds, st, L, vw, h0, f->Ft, f->A, f->N, done);
}

// Layer 0's cell GEMM on B > 1 samples, lifting its rows from (chi, v).
void launch_cell_rows_lift(const cgm_fno* f, hipStream_t st, int rows, const LiftIn& L, const bf16* W,
                           const float* bias, bf16* pre, bf16* out, const int* done) {
  const size_t lds = row_kernel_lds(f->N);
  if (f->N % 4 == 0 && f->N <= 512 && rows / 4 >= 512)
    hipLaunchKernelGGL(k_cell_rows_lift<4>, dim3(rows / 4), dim3(512), lds, st, L, f->Fy, W, f->Bt, bias, pre, out,
                       f->Ft, f->A, f->N, done);
  else if (two_rows(f->N, rows))
    hipLaunchKernelGGL(k_cell_rows_lift<2>, dim3(rows / 2), dim3(512), lds, st, L, f->Fy, W, f->Bt, bias, pre, out,
                       f->Ft, f->A, f->N, done);
  else
    hipLaunchKernelGGL((k_cell_row<false, true>), dim3(rows), dim3(512), lds, st, nullptr, L, f->Fy, W, f->Bt,
                       nullptr, nullptr, bias, pre, out, f->Ft, f->A, f->N, done);
}

// Cell GEMM of layers 0-2 on one sample, B_x from the mixed modes: in pairs
// of rows where single rows would be more blocks than CUs and the pair fits.
void launch_cell_fold(const cgm_fno* f, hipStream_t st, int rows, bool lift, const bf16* P, const LiftIn& L,
                      const bf16* W, const float* bias, bf16* pre, bf16* out, const int* done) {
  if (f->N > 256 && f->N <= 512) {
    auto kern = lift ? k_cell_pair<true> : k_cell_pair<false>;
    hipLaunchKernelGGL(kern, dim3(f->N / 2, rows / f->N), dim3(1024), cell_pair_lds(f->N, lift), st, P, L, f->Fy, W,
                       f->Vm, f->Ex, bias, pre, out, f->Ft, f->A, f->N, done);
  } else {
    auto kern = lift ? k_cell_row<true, true> : k_cell_row<true, false>;
    hipLaunchKernelGGL(kern, dim3(rows), dim3(512), row_kernel_lds(f->N), st, P, L, f->Fy, W, f->Bt, f->Vm, f->Ex,
                       bias, pre, out, f->Ft, f->A, f->N, done);
  }
}

// Cell GEMM of layers 1-2 on B > 1 samples (B_x from R): the most rows per
// work-group (8, 4 or 2) that leave at least 1024 work-groups (4: 512).
void launch_cell_rows(const cgm_fno* f, hipStream_t st, int rows, const bf16* P, const bf16* W, const float* bias,
                      bf16* pre, bf16* out, const int* done) {
  const size_t lds = row_kernel_lds(f->N);
  if (f->N % 8 == 0 && f->N <= 512 && rows / 8 >= 1024)
    hipLaunchKernelGGL(k_cell_rows<8>, dim3(rows / 8), dim3(512), lds, st, P, f->Fy, W, f->Bt, bias, pre, out, f->Ft,
                       f->A, f->N, done);
  else if (f->N % 4 == 0 && f->N <= 512 && rows / 4 >= 512)
    hipLaunchKernelGGL(k_cell_rows<4>, dim3(rows / 4), dim3(512), lds, st, P, f->Fy, W, f->Bt, bias, pre, out, f->Ft,
                       f->A, f->N, done);
  else if (two_rows(f->N, rows))
    hipLaunchKernelGGL(k_cell_rows<2>, dim3(rows / 2), dim3(512), lds, st, P, f->Fy, W, f->Bt, bias, pre, out, f->Ft,
                       f->A, f->N, done);
  else
    hipLaunchKernelGGL((k_cell_row<false, false>), dim3(rows), dim3(512), lds, st, P, LiftIn{}, f->Fy, W, f->Bt,
                       nullptr, nullptr, bias, pre, out, f->Ft, f->A, f->N, done);
}

// Forward pass on B unit-norm vectors (or one lazily normalised vector with
// nrm/vw).  train keeps activations for fno_backward.
int fno_forward_io(cgm_fno* f, hipStream_t st, const FnoIO& io, int B, bool train, const int* done) {
  const float s = (float)f->N;
  const int rows = B * f->N;
  const size_t lds = row_kernel_lds(f->N);
  const bool fold = B == 1;
  int rc;
  LiftIn L{io.chi, io.sChi, f->chi_scale, io.v, io.sV, io.nrm, io.sNrm, s, f->params};
  launch_lift(f, st, rows, L, io.vw, train ? f->h[0] : nullptr, done);
  CGM_HIP(hipGetLastError());
  const float2* vv = io.vw ? io.vw : io.v;
  // layer 0 lifts its rows again from v' (normalised by k_lift_row into vw
  // when given) instead of reading h0
  LiftIn L0 = L;
  if (io.vw) {
    L0.v = io.vw;
    L0.nrm = nullptr;
  }
  for (int l = 0; l < 4; ++l) {
    const float* Lp = f->params + layer_off(l);
    // x-DFT and mixing; for one sample the inverse x-DFT of each row of
    // layers 0-2 runs in its cell GEMM, otherwise k_invx forms every B_x once
    const bool fold_l = fold && l < 3;
    if ((rc = spectral(f, st, (const float2*)(Lp + C * C + C), train ? f->U[l] : nullptr, false, B, done,
                       !fold_l)))
      return rc;
    const bf16* Wl = f->Wt + l * C * C;
    if (l < 3 && (l > 0 || train) && !fold) {  // training has h0 in memory: reading it beats lifting again
      launch_cell_rows(f, st, rows, f->h[l], Wl, Lp + C * C, train ? f->pre[l] : nullptr, f->h[l + 1], done);
    } else if (l == 0 && !fold) {
      launch_cell_rows_lift(f, st, rows, L0, Wl, Lp + C * C, train ? f->pre[0] : nullptr, f->h[1], done);
    } else if (l < 3) {
      launch_cell_fold(f, st, rows, l == 0, f->h[l], L0, Wl, Lp + C * C, train ? f->pre[l] : nullptr, f->h[l + 1],
                       done);
    } else {
      const long waves = (long)B * f->n / 64;
      CGM_CHECK(waves % 4 == 0, CGM_ERROR_UNSUPPORTED, "cell GEMM needs N %% 64 == 0");
      hipLaunchKernelGGL(k_cell_proj, dim3((unsigned)(waves / 4)), dim3(256), 0, st, f->h[3], f->Fy, Wl, f->Bt,
                         Lp + C * C, train ? f->h[4] : nullptr, f->params, vv, io.sV, io.vw ? nullptr : io.nrm,
                         io.sNrm, s, io.z, io.sZ, f->N, done);
    }
    CGM_HIP(hipGetLastError());
  }
  if (train) {
    f->fwd_batch = B;
    f->chi_in = io.chi;
    f->v_in = vv;
  }
  return CGM_SUCCESS;
}

int fno_forward(cgm_fno* f, hipStream_t st, const float* chi, const float2* v, const double* nrm, float2* vw,
                float2* z, int B, bool train, const int* done) {
  FnoIO io;
  io.chi = chi;
  io.sChi = f->n;
  io.v = v;
  io.sV = f->n;
  io.nrm = nrm;
  io.sNrm = 0;
  io.vw = vw;
  io.z = z;
  io.sZ = f->n;
  return fno_forward_io(f, st, io, B, train, done);
}

int fno_batch(const cgm_fno* f) { return f->B; }

cgm_context* fno_context(const cgm_fno* f) { return f->ctx; }

}  // namespace cgm

static int fno_backward(cgm_fno* f, const float2* dz, float* grad) {
  hipStream_t st = f->ctx->stream;
  const int B = f->fwd_batch;
  const long total = (long)B * f->n, nseg = total / 64;  // N % 64 == 0, so nseg % 4 == 0
  const int rows = B * f->N;
  const float s = (float)f->N, is = 1.f / s;
  const float* Wout = f->params + kOffOut;
  int rc;
  // partials of every reduction, summed by one launch at the end
  ReduceList list;
  float* part = f->part;
  int nb = 0, ns = 0;
  auto segment = [&](int G, int width, float* out) {
    float* p = part;
    list.seg[ns++] = ReduceSeg{p, out, G, width, nb};
    nb += (width + 63) / 64;
    part += (size_t)G * width;
    return p;
  };
  SpecGrads sg;
  hipLaunchKernelGGL(k_proj_bwd, dim3(kProjGrid), dim3(256), 0, st, dz, f->h[4], f->v_in, is,
                     segment(kProjGrid, kProjPart, grad + kOffOut), total);
  CGM_HIP(hipGetLastError());
  // layer 3 has no activation: its pre-activation gradient is dh4, which its
  // kernels form from dz
  const bf16* dpre = nullptr;
  for (int l = 3; l >= 0; --l) {
    const float* Lp = f->params + layer_off(l);
    float* Lg = grad + layer_off(l);
    // g_B rows (basis F), dW_l and db_l partials
    if ((rc = launch_back_rows(f, st, dpre, dz, f->h[l], segment(back_rows_grid(rows), kRowPart, Lg), B)))
      return rc;
    // spectral adjoint: dV (saved), dA rows into Bt
    if ((rc = spectral(f, st, (const float2*)(Lp + C * C + C), f->dV[l], true, B, nullptr))) return rc;
    sg.U[l] = f->U[l];
    sg.dV[l] = f->dV[l];
    sg.G[l] = (float2*)(Lg + C * C + C);
    const bf16* Wl = f->Wn + l * C * C;
    bf16* dnext = f->dh[l & 1];
    const dim3 grid((unsigned)(nseg / 4));
    if (l == 3)
      hipLaunchKernelGGL(k_back_cells<true>, grid, dim3(256), 0, st, dpre, dz, Wout, is, f->Fy, Wl, f->Bt,
                         f->pre[l - 1], dnext, f->N);
    else if (l > 0)
      hipLaunchKernelGGL(k_back_cells<false>, grid, dim3(256), 0, st, dpre, dz, Wout, is, f->Fy, Wl, f->Bt,
                         f->pre[l - 1], dnext, f->N);
    else {
      const int G = back_cells_grid(nseg);
      hipLaunchKernelGGL(k_back_lift, dim3(G), dim3(256), 0, st, dpre, f->Fy, Wl, f->Bt, f->chi_in, f->chi_scale,
                         f->v_in, s, segment(G, kLiftPart, grad), f->N, nseg);
    }
    CGM_HIP(hipGetLastError());
    dpre = dnext;
  }
  hipLaunchKernelGGL(k_specgrad, dim3(KX * KY, 4), dim3(256), 0, st, sg, B);
  hipLaunchKernelGGL(k_reduce_part, dim3(nb), dim3(1024), 0, st, list);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

extern "C" int cgm_fno_num_params(size_t* n) {
  CGM_CHECK(n, CGM_ERROR_INVALID_VALUE, "null argument");
  *n = (size_t)kNumParams;
  return CGM_SUCCESS;
}

extern "C" int cgm_fno_create(cgm_ctx_t c, int batch, float chi_scale, cgm_fno_t* out) {
  CGM_CHECK(c && out, CGM_ERROR_INVALID_VALUE, "null argument");
  *out = nullptr;
  CGM_CHECK(batch >= 1, CGM_ERROR_INVALID_VALUE, "batch %d < 1", batch);
  const int N = c->N;
  CGM_CHECK(N >= 64 && N <= 1024 && N % 64 == 0, CGM_ERROR_UNSUPPORTED,
            "the FNO preconditioner needs 64 <= N <= 1024 with N %% 64 == 0 (N = %d)", N);
  CGM_HIP(hipSetDevice(c->device));
  cgm_fno* f = new cgm_fno();
  f->ctx = c;
  f->device = c->device;
  f->N = N;
  f->B = batch;
  f->n = (long)N * N;
  f->chi_scale = chi_scale;
  const size_t act = sizeof(bf16) * (size_t)batch * f->n * C;
  int rc = CGM_SUCCESS;
  auto alloc = [&](void** p, size_t bytes) {
    if (rc) return;
    if (hipMalloc(p, bytes) != hipSuccess) {
      cgm_set_last_error("cgm_fno_create: hipMalloc of %zu bytes failed", bytes);
      rc = CGM_ERROR_ALLOC;
    }
  };
  alloc((void**)&f->Wt, sizeof(bf16) * 4 * C * C);
  alloc((void**)&f->Wn, sizeof(bf16) * 4 * C * C);
  alloc((void**)&f->Ft, sizeof(bf16) * C * N);
  alloc((void**)&f->Fy, sizeof(bf16) * C * N);
  alloc((void**)&f->Ex, sizeof(float2) * KX * N);
  for (int l = 0; l < 5; ++l) alloc((void**)&f->h[l], act);
  for (int l = 0; l < 3; ++l) alloc((void**)&f->pre[l], act);
  for (int l = 0; l < 2; ++l) alloc((void**)&f->dh[l], act);
  alloc((void**)&f->A, sizeof(float) * (size_t)batch * N * C * C);
  for (int l = 0; l < 4; ++l) alloc((void**)&f->U[l], sizeof(float2) * (size_t)batch * KX * KY * C);
  for (int l = 0; l < 4; ++l) alloc((void**)&f->dV[l], sizeof(float2) * (size_t)batch * KX * KY * C);
  alloc((void**)&f->Vm, sizeof(float2) * (size_t)batch * KX * KY * C);
  alloc((void**)&f->Bt, sizeof(bf16) * (size_t)batch * N * C * C);
  alloc((void**)&f->part, sizeof(float) * ((size_t)4 * back_rows_grid(batch * N) * kRowPart +
                                           (size_t)kProjGrid * kProjPart +
                                           (size_t)back_cells_grid(batch * f->n / 64) * kLiftPart));
  if (rc) {
    fno_free(f);
    delete f;
    return rc;
  }
  // column basis and row twiddles (computed in double, stored rounded)
  std::vector<bf16> ft((size_t)C * N), fy((size_t)C * N);
  std::vector<float2> ex((size_t)KX * N);
  for (int y = 0; y < N; ++y) {
    for (int ky = 0; ky < KY; ++ky) {
      const double th = 2.0 * M_PI * (double)((long)ky * y % N) / N;
      const float cs = (float)cos(th), sn = (float)-sin(th);
      ft[(size_t)(2 * ky) * N + y] = (bf16)cs;
      ft[(size_t)(2 * ky + 1) * N + y] = (bf16)sn;
      fy[(size_t)y * C + 2 * ky] = (bf16)cs;
      fy[(size_t)y * C + 2 * ky + 1] = (bf16)sn;
    }
    for (int q = 0; q < KX; ++q) {
      const long kx = q < 16 ? q : N - KX + q;
      const double ph = 2.0 * M_PI * (double)(kx * y % N) / N;
      ex[(size_t)q * N + y] = make_float2((float)cos(ph), (float)sin(ph));
    }
  }
  if (hipMemcpy(f->Ft, ft.data(), sizeof(bf16) * ft.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(f->Fy, fy.data(), sizeof(bf16) * fy.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(f->Ex, ex.data(), sizeof(float2) * ex.size(), hipMemcpyHostToDevice) != hipSuccess) {
    cgm_set_last_error("cgm_fno_create: copy of the bases failed");
    rc = CGM_ERROR_DEVICE;
  }
  if (!rc) rc = lds_limits();
  if (rc) {
    fno_free(f);
    delete f;
    return rc;
  }
  *out = f;
  return CGM_SUCCESS;
}

extern "C" int cgm_fno_destroy(cgm_fno_t f) {
  if (!f) return CGM_SUCCESS;
  (void)hipSetDevice(f->device);
  fno_free(f);
  delete f;
  return CGM_SUCCESS;
}

extern "C" int cgm_fno_set_params(cgm_fno_t f, const float* params) {
  CGM_CHECK(f && params, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(((uintptr_t)params & 15) == 0, CGM_ERROR_INVALID_VALUE, "parameters must be 16-byte aligned");
  CGM_HIP(hipSetDevice(f->ctx->device));
  f->params = params;
  hipLaunchKernelGGL(k_prep, dim3(4 * C * C / 256), dim3(256), 0, f->ctx->stream, params, f->Wt, f->Wn);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

extern "C" int cgm_fno_forward(cgm_fno_t f, const float* chi, const cgm_complex64* v, cgm_complex64* z, int batch,
                               int train) {
  CGM_CHECK(f && chi && v && z, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(f->params, CGM_ERROR_INVALID_VALUE, "cgm_fno_set_params has not been called");
  CGM_CHECK(batch >= 1 && batch <= f->B, CGM_ERROR_INVALID_VALUE, "batch %d outside [1, %d]", batch, f->B);
  CGM_CHECK((const void*)v != (const void*)z, CGM_ERROR_INVALID_VALUE, "v and z must not alias");
  CGM_HIP(hipSetDevice(f->ctx->device));
  return fno_forward(f, f->ctx->stream, chi, (const float2*)v, nullptr, nullptr, (float2*)z, batch, train != 0,
                     nullptr);
}

extern "C" int cgm_fno_backward(cgm_fno_t f, const cgm_complex64* dz, float* grad) {
  CGM_CHECK(f && dz && grad, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(f->fwd_batch > 0, CGM_ERROR_INVALID_VALUE, "cgm_fno_backward needs a preceding training forward");
  CGM_HIP(hipSetDevice(f->ctx->device));
  return fno_backward(f, (const float2*)dz, grad);
}

// Average device time (ms, HIP events on the context stream, reps launches
// after two warm-ups) of each kernel of the network on `batch` vectors
// (contiguous [batch][N*N] chi, v, z): ms[0] lift with the first row projection (k_lift_row),
// [1] row projection with the weight gradient (k_back_rows, the backward pass), [2] x-DFT
// with the mode mixing (k_spectral), [3] unused (0), [4] inverse x-DFT, [5] cell GEMM with GELU and the next row
// projection (k_cell_row of layers 1-2, forming B_x itself for batch 1), [6]
// last cell GEMM with the projection (k_cell_proj), [7] one whole forward
// pass, [8] the cell GEMM of layer 0 (k_cell_row lifting its row from chi
// and v).  The lift of [0] keeps h0 in LDS only, as in inference.
extern "C" int cgm_fno_profile(cgm_fno_t f, const float* chi, const cgm_complex64* v, cgm_complex64* z, int batch,
                               int reps, float* ms) {
  CGM_CHECK(f && chi && v && z && ms && reps > 0, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(batch >= 1 && batch <= f->B, CGM_ERROR_INVALID_VALUE, "batch %d outside [1, %d]", batch, f->B);
  CGM_CHECK(f->params, CGM_ERROR_INVALID_VALUE, "cgm_fno_set_params has not been called");
  CGM_HIP(hipSetDevice(f->ctx->device));
  hipStream_t st = f->ctx->stream;
  const int B = batch;
  const long total = (long)B * f->n;
  const unsigned rows = (unsigned)(B * f->N);
  const float s = (float)f->N;
  const float* Lp = f->params + layer_off(0);
  const float2* W = (const float2*)(Lp + C * C + C);
  const size_t lds = row_kernel_lds(f->N);
  hipEvent_t e0, e1;
  CGM_HIP(hipEventCreate(&e0));
  CGM_HIP(hipEventCreate(&e1));
  const LiftIn L{chi, f->n, f->chi_scale, (const float2*)v, f->n, nullptr, 0L, s, f->params};
  int rc = CGM_SUCCESS;
  for (int k = 0; k < 9 && !rc; ++k) {
    for (int r = -2; r < reps && !rc; ++r) {
      if (r == 0) CGM_HIP(hipEventRecord(e0, st));
      switch (k) {
        case 3: break;
        case 0:  // the first warm-up also stores h0, which cases 1 and 5 read
          launch_lift(f, st, rows, L, nullptr, r == -2 ? f->h[0] : nullptr, nullptr);
          break;
        case 1: rc = launch_back_rows(f, st, f->h[0], nullptr, f->h[1], f->part, B); break;
        case 2: launch_spectral(f, st, W, nullptr, false, B, nullptr); break;
        case 4:
          launch_invx(f, st, B, nullptr);
          break;
        case 5:
          if (B == 1)
            launch_cell_fold(f, st, rows, false, f->h[0], L, f->Wt, Lp + C * C, nullptr, f->h[1], nullptr);
          else
            launch_cell_rows(f, st, rows, f->h[0], f->Wt, Lp + C * C, nullptr, f->h[1], nullptr);
          break;
        case 8:
          if (B == 1)
            launch_cell_fold(f, st, rows, true, nullptr, L, f->Wt, Lp + C * C, nullptr, f->h[1], nullptr);
          else
            launch_cell_rows_lift(f, st, rows, L, f->Wt, Lp + C * C, nullptr, f->h[1], nullptr);
          break;
        case 6:
          hipLaunchKernelGGL(k_cell_proj, dim3((unsigned)(total / 256)), dim3(256), 0, st, f->h[3], f->Fy, f->Wt,
                             f->Bt, Lp + C * C, nullptr, f->params, (const float2*)v, f->n, nullptr, 0L, s,
                             (float2*)z, f->n, f->N, nullptr);
          break;
        default:
          rc = fno_forward(f, st, chi, (const float2*)v, nullptr, nullptr, (float2*)z, B, false, nullptr);
          break;
      }
      if (hipGetLastError() != hipSuccess) rc = CGM_ERROR_DEVICE;
    }
    CGM_HIP(hipEventRecord(e1, st));
    CGM_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    CGM_HIP(hipEventElapsedTime(&t, e0, e1));
    ms[k] = k == 3 ? 0.f : t / reps;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}
