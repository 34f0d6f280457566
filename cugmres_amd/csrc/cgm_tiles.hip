// Tile (block-Jacobi) right preconditioner: exact inverses of the operator
// restricted to square tiles of the grid.
//
// The reference has no preconditioner (B/CUDA_GMRES/GMRES.cuh:22-446 runs
// plain GMRES).  On the high-contrast maps of the benchmark workloads
// (eps in {1, 12.1}, h = lambda/20) GMRES needs a number of steps that grows
// about as N^1.8 (335 at N = 64, 1,155 at N = 128 unrestarted), because every
// high-permittivity block is a near-resonant scatterer.  Inverting the
// operator exactly on T x T tiles removes those local resonances.
//
// On tile t (cells (a T + r, b T + c), 0 <= r, c < T, row-major inside the
// tile) the local operator is
//     A_t = I - G_t diag(chi_t),   G_t[p, q] = g[|p_r - q_r|, |p_c - q_c|],
// with g the N x N generator block of the operator (the block whose circulant
// embedding gives the kernel spectrum).
//
// Tiles of side 8, 16, 32 (dense form): every A_t is formed in FP32 complex
// (column-major, T^2 x T^2) and inverted in place by a batched LU with
// partial pivoting (rocSOLVER getrf + getri), once per map.  Application, once
// per Krylov step: y_t = A_t^{-1} x_t, one work-group per (tile, system), one
// thread per output cell streaming its row of the inverse column by column
// (coalesced: the inverse is column-major), the tile's input staged in LDS.
// A map shared by several right-hand sides is factored once, and each
// work-group then applies its tile's inverse to all of them while it streams
// it.
//
// Tiles of side 64 and 128 (reduced form).  With S the cells of the tile
// where chi != 0 and D_S = diag(chi_S), the columns of A_t outside S are unit
// vectors, and
//     A_t^{-1} = I + G_t[:, S] W_t R_S,   W_t = (I - D_S G_SS)^{-1} D_S
// (R_S restricts to S).  Factorisation inverts only the |S| x |S| matrices
// D_S^{-1} - G_SS = D_S^{-1} (I - D_S G_SS), whose inverse is W_t (a symmetric
// block sweep with rocBLAS updates and an LDS pivot-block kernel), and keeps
// W_t in FP16 complex, scaled per tile by its largest magnitude.  Application:
// u_t = W_t x_t[S] (the only large stream: W_t is complex symmetric, since
// W_t = (D_S^{-1} - G_SS)^{-1}, and only the lower triangle of its 128 x 128
// blocks is stored and streamed), then G_t u_t for all tiles at once as a
// batch of T x T convolutions through the operator's own FFT passes at size
// 2T with the tile's spectrum, the last of which adds x: y = x + G_t u_t.  On the benchmark maps
// 3/8 of the cells carry chi != 0, so a 128 x 128 tile streams about 4 % of
// the entries of its dense inverse, and the inversion work drops by about
// 20x; that makes 128 x 128 tiles affordable, which take 1,032 Krylov steps
// on seed 0 at N = 512 against 2,380 for 64 x 64 and 4,573 for 32 x 32.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <map>
#include <type_traits>
#include <vector>

#include "cgm_fft.h"
#include "cgm_internal.h"
#include "cgm_special.h"

using namespace cgm;

// One work-group's share of a tile's W (k_tile_ws): block column j0 (and j0 + 1)
// and the block rows from i0 on.
struct Strip {
  long woff;   // the tile's first block in W16
  int bloc;    // the tile's first block row among its map's
  int nB;      // block rows of the tile
  int i0, j0;
};
// Strips of two block columns and several rows, of two columns and one row, of
// one column and one row.
enum StripKind { kLongStrip, kRowStrip, kBlockStrip };

struct cgm_tiles {
  cgm_context* ctx = nullptr;
  int device = 0;
  int N = 0, T = 0, B = 0;  // grid, tile side, systems (maps) the workspace holds
  int nt = 0;               // tiles per grid side
  int M2 = 0;               // unknowns per tile (T * T)
  bool reduced = false;     // T >= 64: reduced form
  int maps = 0;             // maps factored by the last cgm_tiles_factor (1: shared)
  bool maps1 = true;        // the layout below is that of one map
  rocblas_handle h = nullptr;
  size_t bytes = 0;         // device memory held
  // dense form (T <= 32)
  float2* K = nullptr;       // [B][nt * nt][M2 * M2] inverses, column-major
  int* ipiv = nullptr;      // [B][nt * nt][M2]
  int* info = nullptr;      // [B][nt * nt]       (reduced form: singular-pivot flags)
  // reduced form (T >= 64)
  int* ncol = nullptr;             // [B][nt * nt] |S_t| padded to a multiple of kPadTo
  unsigned short* cols = nullptr;  // [B][nt * nt][M2] the cells of S_t in order, then kPadCol
  long* woff = nullptr;            // [B][nt * nt] offset of W_t in W16 (half2 elements)
  float* kscale = nullptr;         // [B][nt * nt] largest |W_t| entry
  int* ids = nullptr;              // [B][nt * nt] factor members (tiles with n_t > 0), by size
  int* bloc = nullptr;             // [B][nt * nt] each tile's first block row among its map's
  int* sloc = nullptr;             // [B][nt * nt] each tile's first entry in spos
  Strip* stab = nullptr;           // strip lists of the maps, largest first
  int* spos = nullptr;             // by tile, [si][64]: place of strip (si, sj) in the map's list
  size_t stab_cap = 0, spos_cap = 0;
  int* sstart = nullptr;           // [B] first entry of each map's list in stab
  int* scount = nullptr;           // [B] strips of each map
  int* ssize = nullptr;            // [B] block rows of a map's strips and, << 8, their block columns
  int scount_max = 0;              // largest strip count over the factored maps
  unsigned kinds = 0;              // which StripKinds the maps have (bits)
  long plen_max = 0;               // largest scount * (columns + rows of a strip)
  int xblk_max = 0;                // largest number of block rows of a map
  int nbmax = 0;                   // largest number of block rows of a tile
  float4* Pw = nullptr;            // [group][strip][columns, rows][64 systems of the group] partial products (apply)
  size_t pw_cap = 0;
  unsigned* Xs = nullptr;          // [group][xblk_max][kXsBlk] inputs in FP16 parts (apply)
  size_t xs_cap = 0;
  float* xinv = nullptr;           // [sys][nt * nt] inverse scales of the inputs (apply)
  size_t xinv_cap = 0;
  long* koff = nullptr;            // [B][nt * nt] offset of each member's matrix in Kw
  int* nl = nullptr;               // [B][nt * nt] each member's matrix side (n_t padded to kBlk)
  __half2* W16 = nullptr;          // W_t / kscale_t in FP16: the kBlkW x kBlkW blocks (i, j <= i) of the
                                   // lower triangle, each column-major, row-major over the blocks
  size_t w16_cap = 0;              // elements
  float2* Kw = nullptr;            // FP32 matrices of the members (factor)
  size_t kw_cap = 0;               // elements
  float2* Pb = nullptr;            // [member][kBlk][kBlk] pivot blocks (factor)
  size_t pb_cap = 0;
  float2* Rw = nullptr;            // kBlk x n_max row block (factor)
  size_t rw_cap = 0;
  float2* Cw = nullptr;            // n_max x kBlk column block (factor)
  size_t cw_cap = 0;
  float2* U = nullptr;             // [sys][nt * nt][M2] u_t scattered on the tile (apply)
  float2* Tm = nullptr;            // [sys][nt * nt][T * 2T] FFT scratch (apply)
  int scratch_sys = 0;             // systems the apply scratch holds
  Plan P;                          // tile convolution: N' = T, M' = 2T
  float2* tw32 = nullptr;          // twiddles of size M'
  double2* tw64 = nullptr;
  double2* blkT = nullptr;         // T x T corner of the generator block
  float2* gq = nullptr;            // quarter spectrum of the tile convolution
  std::vector<double> kept;        // per map: inverse entries streamed per application
};

namespace {

constexpr int kBuildChunk = 65536;           // matrix entries per work-group of the build kernels
constexpr int kPadTo = 16;                   // n_t is padded to a multiple of this
constexpr unsigned short kPadCol = 0xFFFF;   // cell index of a padding slot
constexpr int kBlk = 128;                    // block of the Gauss-Jordan inversion (reduced form)
constexpr int kBlkW = 128;                   // block of the symmetric storage of W (apply)
constexpr int kSplits = 3;                   // FP16 parts of one FP32 input value (apply)
constexpr int kXsBlk = kSplits * 16 * kBlkW; // dwords of one block row's inputs in Xs (apply)

template <typename P>
int grow(cgm_tiles* t, P** p, size_t* cap, size_t need) {
  if (need <= *cap) return CGM_SUCCESS;
  if (*p) {
    (void)hipFree(*p);
    t->bytes -= *cap * sizeof(P);
    *p = nullptr;
    *cap = 0;
  }
  if (hipMalloc((void**)p, need * sizeof(P)) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();  // the caller reports it; the next launch's check must not
    cgm_set_last_error("tile preconditioner: allocation of %zu MiB failed", need * sizeof(P) >> 20);
    return CGM_ERROR_ALLOC;
  }
  *cap = need;
  t->bytes += need * sizeof(P);
  return CGM_SUCCESS;
}

// ---------------------------------------------------------------------------
// dense form (T <= 32)
// ---------------------------------------------------------------------------

// A_t of map blockIdx.y, column-major into K: work-group blockIdx.x covers
// chunk (blockIdx.x % chunks) of tile (blockIdx.x / chunks).
__global__ void __launch_bounds__(256)
k_tile_build(const double2* __restrict__ g, const float* __restrict__ chi, long chi_stride, float2* __restrict__ K,
             int N, int T, int chunks) {
  const int nt = N / T;
  const int M2 = T * T;
  const int t = blockIdx.x / chunks;
  const long e0 = (long)(blockIdx.x % chunks) * kBuildChunk;
  const long e1 = e0 + kBuildChunk < (long)M2 * M2 ? e0 + kBuildChunk : (long)M2 * M2;
  const int a = t / nt, b = t % nt;
  chi += (long)blockIdx.y * chi_stride;
  float2* A = K + ((long)blockIdx.y * nt * nt + t) * (long)M2 * M2;
  for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
    const int p = e % M2, q = e / M2;  // row p, column q
    const int pr = p / T, pc = p % T, qr = q / T, qc = q % T;
    const int dr = pr > qr ? pr - qr : qr - pr;
    const int dc = pc > qc ? pc - qc : qc - pc;
    const double2 gv = g[(long)dr * N + dc];
    const double cq = chi[(long)(a * T + qr) * N + b * T + qc];
    A[e] = make_float2((float)((p == q ? 1.0 : 0.0) - gv.x * cq), (float)(-gv.y * cq));
  }
}

// y_t = K_t x_t for NV vectors that share the tile's inverse (one map) or
// one vector per map (NV = 1).  System s reads io.v + s sV, scaled by 1 /
// *(io.nrm + s sNrm bytes) when io.nrm is given (the scaled input is written to
// io.vw + s sV when io.vw is given), writes io.z + s sZ, and is skipped once
// *(done + s sd bytes) is set.
//
// Tiles of side 8: one wave per tile (blockIdx.x) and group of NV systems
// (blockIdx.y), one row per lane.  Splitting a tile's 64 columns over waves, as
// k_tile_apply does below, costs more than it gives there (N = 512, four
// systems: 25.6 against 28.0 us).
template <int NV>
__global__ void __launch_bounds__(64)
k_tile_apply8(const float2* __restrict__ K, long sK, FnoIO io, const int* __restrict__ done, long sd, int N, int T,
              int nsys) {
  constexpr int M2 = 64;
  constexpr int kU = 8;  // columns of the inverse loaded ahead
  __shared__ float2 xs[NV][M2];
  const int nt = N / T;
  const int t = blockIdx.x;
  const int a = t / nt, b = t % nt;
  const int s0 = blockIdx.y * NV;
  const int r = threadIdx.x;
  const long cell = (long)(a * T + r / T) * N + b * T + r % T;
  bool live[NV];
  bool any = false;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int s = s0 + v;
    live[v] = s < nsys && !(done && *boff(done, (long)s * sd));
    any |= live[v];
    float2 xv = make_float2(0.f, 0.f);
    if (live[v]) {
      xv = io.v[(long)s * io.sV + cell];
      if (io.nrm) {
        const double d = *boff(io.nrm, (long)s * io.sNrm);
        const float sc = d > 0.0 ? (float)(1.0 / d) : 0.f;
        xv.x *= sc;
        xv.y *= sc;
        if (io.vw) io.vw[(long)s * io.sV + cell] = xv;
      }
    }
    xs[v][r] = xv;
  }
  if (!any) return;  // uniform over the work-group
  __syncthreads();
  const float2* Kt = K + (long)(NV == 1 ? s0 : 0) * sK + (long)t * M2 * M2 + r;
  float2 acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = make_float2(0.f, 0.f);
#pragma unroll 2
  for (int q0 = 0; q0 < M2; q0 += kU) {
    float2 k[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) k[u] = Kt[(long)(q0 + u) * M2];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const float2 xv = xs[v][q0 + u];
        acc[v].x += k[u].x * xv.x - k[u].y * xv.y;
        acc[v].y += k[u].x * xv.y + k[u].y * xv.x;
      }
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v)
    if (live[v]) io.z[(long)(s0 + v) * io.sZ + cell] = acc[v];
}

// io.vw = io.v over its norm, system blockIdx.y, before an application that is
// to normalise its input in place: several work-groups of k_tile_apply read a
// tile, so none of them can write to it (a late one would divide again).
__global__ void __launch_bounds__(256)
k_tile_scale(FnoIO io, const int* __restrict__ done, long sd, long n) {
  const int s = blockIdx.y;
  if (done && *boff(done, (long)s * sd)) return;
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  const double d = *boff(io.nrm, (long)s * io.sNrm);
  const float sc = d > 0.0 ? (float)(1.0 / d) : 0.f;
  float2 x = io.v[(long)s * io.sV + e];
  x.x *= sc;
  x.y *= sc;
  io.vw[(long)s * io.sV + e] = x;
}

// Tiles of side 16 and 32: a work-group takes a tile, a block of 128 of its rows
// and a group of NV systems.  io.vw must not be io.v (k_tile_scale).
//
// The stream of K bounds it (8 T^4 bytes per tile; column-major, so rows are
// independent and a row block needs no sum with another).  A wave reads two
// rows per lane (1 KB of a column per load) of every eighth group of four
// columns, kU loads ahead, each register loaded again as soon as it is used and
// not at all in the last round; the waves' sums meet in LDS.  Eight waves on 128
// rows, instead of one thread per row through all columns, keep 16 waves per CU
// on 256 tiles of side 16 where there were four, and 64 tiles of side 32 on all
// CUs.
//
// Work-groups L, L + 8, L + 16.. run on one XCD one after the other: they take the
// groups of systems of one row block (up to 16 per blockIdx.y, so that its L2
// serves all but the first), then the tile's other row blocks.  In the order
// (row block, then tile; groups in blockIdx.y) the second group read K from memory
// again: N = 256, T = 16, nine systems 45 us, now 33.5; T = 32, sixteen 198, now
// 126.  `units` are tiles, or pairs (map, tile) of systems with their own maps
// (NV = 1); fewer than eight would leave XCDs idle, so their row blocks are dealt
// out over the XCDs instead (T = 32, four tiles, one system: 14.0 us on four XCDs,
// 12.2 on eight).
//
// NTL: inverses beyond the 256 MB of Infinity Cache that are read once, without
// a place in the caches (N = 512, T = 16, one system: 91 -> 79 us; N = 384, 302 MB:
// 45.9 -> 44.7; N = 352, 254 MB, is faster with: 36.4 against 37.7).
//
// One / four / sixteen systems of one map, us, against one thread per row: N = 256,
// T = 16 (134 MB): 20.4 / 30.6 / 43.0, here 20.1 / 21.7 / 32.6; N = 512, T = 16 (537
// MB): 91 / 102 / 388, here 79 / 85 / 146; N = 256, T = 32 (537 MB): 201 / 209 / 190,
// here 78 / 81 / 126.  At N = 320, T = 16 (800 work-groups, 3.1 per CU) one system is
// 1.5 us behind it (29.9, here 31.4).  kU = 16 and 4 for up to four systems: 20.5 and
// 20.4 at N = 256, T = 16, 31.5 and 32.4 at N = 320.
constexpr int kTileWaves = 8;
template <int M2, int NV, bool NTL>
__global__ void __launch_bounds__(64 * kTileWaves)
k_tile_apply(const float2* __restrict__ K, long sK, FnoIO io, const int* __restrict__ done, long sd, int N, int T,
             int nsys, int units, int ngroups) {
  constexpr int kWaves = kTileWaves;
  constexpr int RB = 128, kBlocks = M2 / RB;
  constexpr int kUnit = 4;  // loads of one turn of a wave
  constexpr int kU = 8;     // loads ahead: two turns
  static_assert(M2 % (kU * kWaves) == 0, "whole rounds of loads");
  constexpr size_t kXsLen = sizeof(float2) * M2 * NV, kRedLen = sizeof(float4) * (kWaves / 2) * NV * 64;
  __shared__ __align__(16) unsigned char smem[kXsLen > kRedLen ? kXsLen : kRedLen];  // the inputs, then the waves' sums
  float2(*xs)[NV] = reinterpret_cast<float2(*)[NV]>(smem);
  float4(*red)[NV][64] = reinterpret_cast<float4(*)[NV][64]>(smem);
  const int nt = N / T;
  const int xcd = blockIdx.x & 7, step = blockIdx.x >> 3;
  const int row = NV > 1 ? step / ngroups : step;  // row blocks before this one on the XCD
  const int u = units < 8 ? (row * 8 + xcd) / kBlocks : row / kBlocks * 8 + xcd;
  const int rb = (units < 8 ? row * 8 + xcd : row) % kBlocks;
  const int t = NV > 1 ? u : u % (nt * nt);
  const int s0 = NV > 1 ? (blockIdx.y * ngroups + step % ngroups) * NV : u / (nt * nt);
  if (u >= units || s0 >= nsys) return;
  const int a = t / nt, b = t % nt;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  bool live[NV];
  bool any = false;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int s = s0 + v;
    live[v] = s < nsys && !(done && *boff(done, (long)s * sd));
    any |= live[v];
  }
  if (!any) return;  // uniform over the work-group
  const float4* Kt = reinterpret_cast<const float4*>(K + (long)(NV == 1 ? s0 : 0) * sK + (long)t * M2 * M2 + rb * RB) + lane;
  typedef float f4v __attribute__((ext_vector_type(4)));
  const auto load = [&](int q) {  // rows 2 lane, + 1
    const f4v* p = reinterpret_cast<const f4v*>(Kt + (long)q * (M2 / 2));
    if constexpr (NTL) return __builtin_nontemporal_load(p);
    else return *p;
  };
  f4v k[kU];
  // load u of a round: the wave's turns come in the same order for every NV, so
  // a system's sums do not depend on the others
  constexpr int kStep = kU * kWaves;
  const auto col = [&](int u) { return (u / kUnit * kWaves + w) * kUnit + u % kUnit; };
#pragma unroll
  for (int u = 0; u < kU; ++u) k[u] = load(col(u));
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int s = s0 + v;
    float sc = 1.f;
    if (live[v] && io.nrm) {
      const double d = *boff(io.nrm, (long)s * io.sNrm);
      sc = d > 0.0 ? (float)(1.0 / d) : 0.f;
    }
#pragma unroll 1
    for (int r = threadIdx.x; r < M2; r += 64 * kWaves) {
      const long cell = (long)(a * T + r / T) * N + b * T + r % T;
      float2 xv = make_float2(0.f, 0.f);
      if (live[v]) {
        xv = io.v[(long)s * io.sV + cell];
        if (io.nrm) {
          xv.x *= sc;
          xv.y *= sc;
          if (io.vw && rb == 0) io.vw[(long)s * io.sV + cell] = xv;
        }
      }
      xs[r][v] = xv;
    }
  }
  __syncthreads();
  float4 acc[NV];  // the two rows
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = make_float4(0.f, 0.f, 0.f, 0.f);
  const auto add_column = [&](int q, f4v c) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const float2 xv = xs[q][v];
      // two fused multiply-adds each (a product of its own and an addition otherwise)
      acc[v].x = fmaf(-c[1], xv.y, fmaf(c[0], xv.x, acc[v].x));
      acc[v].y = fmaf(c[1], xv.x, fmaf(c[0], xv.y, acc[v].y));
      acc[v].z = fmaf(-c[3], xv.y, fmaf(c[2], xv.x, acc[v].z));
      acc[v].w = fmaf(c[3], xv.x, fmaf(c[2], xv.y, acc[v].w));
    }
  };
  int q = 0;
#pragma unroll 1
  for (; q < M2 - kStep; q += kStep)
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      add_column(q + col(u), k[u]);
      k[u] = load(q + kStep + col(u));
      if (u % 2) __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of their use
    }
#pragma unroll
  for (int u = 0; u < kU; ++u) add_column(q + col(u), k[u]);
  // sums of the eight waves: the upper four to the lower four, then those four
  const auto add = [](float4& o, const float4& p) {
    o.x += p.x;
    o.y += p.y;
    o.z += p.z;
    o.w += p.w;
  };
  __syncthreads();  // the inputs are read
  if (w >= kWaves / 2)
#pragma unroll
    for (int v = 0; v < NV; ++v) red[w - kWaves / 2][v][lane] = acc[v];
  __syncthreads();
  if (w < kWaves / 2)
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      add(acc[v], red[w][v][lane]);
      red[w][v][lane] = acc[v];
    }
  __syncthreads();
  for (int e = threadIdx.x; e < NV * 64; e += 64 * kWaves) {
    const int v = e / 64, l = e % 64;
    const int s = s0 + v;
    if (s >= nsys || (done && *boff(done, (long)s * sd))) continue;
    float4 o = red[0][v][l];
#pragma unroll
    for (int u = 1; u < kWaves / 2; ++u) add(o, red[u][v][l]);
    const int r = rb * RB + 2 * l;  // T is even: the two rows are neighbours on the grid
    const long cell = (long)(a * T + r / T) * N + b * T + r % T;
    float2* z = io.z + (long)s * io.sZ + cell;
    z[0] = make_float2(o.x, o.y);
    z[1] = make_float2(o.z, o.w);
  }
}

// Systems per pass over the inverses of one map.
int dense_group(int M2, int nsys) {
  if (M2 == 64) return nsys > 1 ? 4 : 1;
  return nsys > 4 ? 8 : nsys > 2 ? 4 : nsys;
}

template <int M2>
int launch_apply_m(const cgm_tiles* tl, hipStream_t st, const FnoIO& io, const int* done, long sd, int nsys) {
  const long sK = (long)tl->nt * tl->nt * M2 * M2;
  const int ntiles = tl->nt * tl->nt;
  const int nv = tl->maps == 1 ? dense_group(M2, nsys) : 1;
  const int groups = (nsys + nv - 1) / nv;
  if constexpr (M2 == 64) {
    if (nv == 4)
      hipLaunchKernelGGL(k_tile_apply8<4>, dim3(ntiles, groups), dim3(64), 0, st, tl->K, 0L, io, done, sd, tl->N, tl->T, nsys);
    else
      hipLaunchKernelGGL(k_tile_apply8<1>, dim3(ntiles, groups), dim3(64), 0, st, tl->K, sK, io, done, sd, tl->N, tl->T, nsys);
  } else {
    FnoIO in = io;
    if (io.nrm && io.vw == io.v) {
      const long n = (long)tl->N * tl->N;
      hipLaunchKernelGGL(k_tile_scale, dim3((unsigned)((n + 255) / 256), nsys), dim3(256), 0, st, io, done, sd, n);
      in.nrm = nullptr;
      in.vw = nullptr;
    }
    // every entry read once, and more of them than the Infinity Cache holds
    const size_t bytes = sizeof(float2) * sK * (tl->maps == 1 ? 1 : nsys);
    const bool ntl = (tl->maps > 1 || groups == 1) && bytes > (size_t)256 << 20;
    const int units = nv > 1 ? ntiles : ntiles * groups, ng = nv > 1 ? std::min(groups, 16) : 1;
    const dim3 grid((units + 7) / 8 * 8 * (M2 / 128) * ng, nv > 1 ? (groups + ng - 1) / ng : 1);
#define CGM_DENSE(NV, S)                                                                                             \
  hipLaunchKernelGGL((ntl ? k_tile_apply<M2, NV, true> : k_tile_apply<M2, NV, false>), grid, dim3(64 * kTileWaves), 0, \
                     st, tl->K, S, in, done, sd, tl->N, tl->T, nsys, units, ng)
    switch (nv) {
      case 8: CGM_DENSE(8, 0L); break;
      case 4: CGM_DENSE(4, 0L); break;
      case 2: CGM_DENSE(2, 0L); break;
      default: CGM_DENSE(1, sK); break;
    }
#undef CGM_DENSE
  }
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

// ---------------------------------------------------------------------------
// reduced form (T = 64, 128): factorisation
// ---------------------------------------------------------------------------

// S_t of every tile of map blockIdx.y (tile blockIdx.x): the cells with
// chi != 0 in row-major order and their count padded to kPadTo (padding
// slots hold kPadCol).
template <int T>
__global__ void __launch_bounds__(1024)
k_tile_cols(const float* __restrict__ chi, long chi_stride, int N, int* __restrict__ ncol,
            unsigned short* __restrict__ cols) {
  constexpr int M2 = T * T;
  constexpr int CPT = M2 / 1024;  // cells per thread
  const int nt = N / T;
  const int t = blockIdx.x, a = t / nt, b = t % nt;
  const long tb = (long)blockIdx.y * nt * nt + t;
  chi += (long)blockIdx.y * chi_stride;
  __shared__ int wsum[16];
  bool nz[CPT];
  int cnt = 0;
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = CPT * threadIdx.x + i;
    nz[i] = chi[(long)(a * T + c / T) * N + b * T + c % T] != 0.f;
    cnt += nz[i];
  }
  // exclusive scan of the counts over the work-group (16 waves of 64)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wave; ++w) base += wsum[w];
  int slot = base + inc - cnt;
  unsigned short* ct = cols + tb * M2;
#pragma unroll
  for (int i = 0; i < CPT; ++i)
    if (nz[i]) ct[slot++] = (unsigned short)(CPT * threadIdx.x + i);
  int total = 0;
  for (int w = 0; w < 16; ++w) total += wsum[w];
  const int padded = (total + kPadTo - 1) / kPadTo * kPadTo;
  if ((int)threadIdx.x < padded - total) ct[total + threadIdx.x] = kPadCol;
  if (threadIdx.x == 0) ncol[tb] = padded;
}

// Grid index of cell c (row-major inside the tile) of tile t.
__device__ inline long tile_cell(int t, int c, int nt, int T, int N) {
  const int a = t / nt, b = t % nt;
  return (long)(a * T + c / T) * N + b * T + c % T;
}

// A = D_S^{-1} - G_SS of member blockIdx.y (tile ids[.]) into Kw + koff[.],
// nl x nl column-major, the identity on padding slots and beyond n_t (A is
// complex symmetric: G is, D_S is real diagonal; W_t = A^{-1}); work-group
// blockIdx.x covers one chunk of the entries.
__global__ void __launch_bounds__(256)
k_tile_build_red(const double2* __restrict__ g, const float* __restrict__ chi, long chi_stride,
                 const int* __restrict__ ncol, const unsigned short* __restrict__ cols, const int* __restrict__ ids,
                 const long* __restrict__ koff, const int* __restrict__ nl, float2* __restrict__ Kw, int N, int T) {
  const int nt = N / T;
  const int i = blockIdx.y;
  const int n = nl[i];
  const long nn = (long)n * n;
  const long e0 = (long)blockIdx.x * kBuildChunk;
  if (e0 >= nn) return;
  const long e1 = e0 + kBuildChunk < nn ? e0 + kBuildChunk : nn;
  const int tb = ids[i];
  const int map = tb / (nt * nt), t = tb % (nt * nt);
  const int nk = ncol[tb];
  const unsigned short* ct = cols + (long)tb * T * T;
  chi += (long)map * chi_stride;
  float2* A = Kw + koff[i];
  for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
    const int p = (int)(e % n), q = (int)(e / n);
    const int cp = p < nk ? ct[p] : kPadCol, cq = q < nk ? ct[q] : kPadCol;
    float2 v = make_float2(p == q ? 1.f : 0.f, 0.f);
    if (cp != kPadCol && cq != kPadCol) {
      const int pr = cp / T, pc = cp % T, qr = cq / T, qc = cq % T;
      const int dr = pr > qr ? pr - qr : qr - pr;
      const int dc = pc > qc ? pc - qc : qc - pc;
      const double2 gv = g[(long)dr * N + dc];
      const double d = p == q ? 1.0 / (double)chi[tile_cell(t, cp, nt, T, N)] : 0.0;
      v = make_float2((float)(d - gv.x), (float)(-gv.y));
    }
    A[e] = v;
  }
}

// Pb[i] = the symmetric kBlk x kBlk diagonal block at k0 of member i
// (column-major), mirrored from the lower triangle where the sweep keeps it.
__global__ void __launch_bounds__(256)
k_gj_gather(const float2* __restrict__ Kw, const long* __restrict__ koff, const int* __restrict__ nl, int k0,
            float2* __restrict__ Pb) {
  const int i = blockIdx.x;
  const int n = nl[i];
  const float2* M = Kw + koff[i];
  float2* P = Pb + (long)i * kBlk * kBlk;
  for (int e = threadIdx.x; e < kBlk * kBlk; e += blockDim.x) {
    const int r = e % kBlk, c = e / kBlk;
    const int hi = r > c ? r : c, lo = r > c ? c : r;
    P[e] = M[(long)(k0 + lo) * n + k0 + hi];
  }
}

// Column block C (n x kBlk, column-major) of pivot block k0 of one member's
// symmetric matrix M (lower triangle kept): rows i < k0 from the row block
// (M(k0 + c, i)), rows in the pivot block mirrored, rows i >= k0 + kBlk from
// the column block (M(i, k0 + c)).  32 x 32 tiles through LDS, so that the
// transposed part reads and writes along columns.
__global__ void __launch_bounds__(256)
k_sw_gather(const float2* __restrict__ M, int n, int k0, float2* __restrict__ C) {
  __shared__ float2 tile[32][33];
  const int i0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int k = ty; k < 32; k += 8) {
    // tile[a][b] = C(i0 + a, c0 + b), every read along a column of M
    if (i0 < k0) {  // C(i0 + k, c0 + tx) = M(k0 + c0 + tx, i0 + k): column i0 + k, contiguous in tx
      tile[k][tx] = M[(long)(i0 + k) * n + k0 + c0 + tx];
    } else {
      const int i = i0 + tx, c = k0 + c0 + k;  // C(i, c - k0) = M(max, min) of (i, c)
      const int hi = i > c ? i : c, lo = i > c ? c : i;
      tile[tx][k] = M[(long)lo * n + hi];
    }
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) C[(long)(c0 + k) * n + i0 + tx] = tile[tx][k];
}

// Writes back the swept column block: CP = C P (n x kBlk) goes to rows
// i >= k0 + kBlk of the column block and, transposed, to the row block for
// rows i < k0; the pivot block becomes -P (its lower triangle is used).
__global__ void __launch_bounds__(256)
k_sw_scatter(float2* __restrict__ M, int n, int k0, const float2* __restrict__ CP, const float2* __restrict__ P) {
  __shared__ float2 tile[32][33];
  const int i0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  if (i0 >= k0 && i0 < k0 + kBlk) {  // the pivot block: -P
    for (int k = ty; k < 32; k += 8) {
      const float2 v = P[(long)(c0 + k) * kBlk + i0 - k0 + tx];
      M[(long)(k0 + c0 + k) * n + i0 + tx] = make_float2(-v.x, -v.y);
    }
    return;
  }
  if (i0 >= k0) {  // below: column block, straight copy along columns
    for (int k = ty; k < 32; k += 8) M[(long)(k0 + c0 + k) * n + i0 + tx] = CP[(long)(c0 + k) * n + i0 + tx];
    return;
  }
  for (int k = ty; k < 32; k += 8) tile[k][tx] = CP[(long)(c0 + k) * n + i0 + tx];  // CP(i0 + tx, c0 + k)
  __syncthreads();
  // M(k0 + c0 + tx, i0 + k) = CP(i0 + k, c0 + tx): column i0 + k of M, contiguous in tx
  for (int k = ty; k < 32; k += 8) M[(long)(i0 + k) * n + k0 + c0 + tx] = tile[tx][k];
}

// In-place inverse of the kBlk x kBlk block Pb[blockIdx.x] (column-major) by
// Gauss-Jordan elimination with partial (row) pivoting in LDS: at step j the
// largest |A(i, j)|, i >= j, is swapped into row j, row j is divided by the
// pivot (its diagonal entry taking the pivot's inverse), every other row i
// loses A(i, j) times row j (its column-j entry taking -A(i, j) / pivot), and
// the row swaps are undone as column swaps in reverse order at the end.
// info[blockIdx.x] is set when a pivot is zero.
__global__ void __launch_bounds__(1024) k_gj_inv(float2* __restrict__ Pb, int* __restrict__ info) {
  constexpr int L = kBlk, LP = kBlk + 1;  // LDS column stride padded against bank conflicts
  __shared__ float2 A[L * LP];
  __shared__ float2 f[L];
  __shared__ int perm[L];
  __shared__ int sp;
  float2* P = Pb + (long)blockIdx.x * L * L;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < L * L; e += blockDim.x) A[(e / L) * LP + e % L] = P[e];
  __syncthreads();
  bool bad = false;
  for (int j = 0; j < L; ++j) {
    if (wave == 0) {
      float best = -1.f;
      int bi = j;
      for (int i = j + lane; i < L; i += 64) {
        const float2 v = A[j * LP + i];
        const float m = v.x * v.x + v.y * v.y;
        if (m > best) {
          best = m;
          bi = i;
        }
      }
      for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (lane == 0) {
        sp = bi;
        perm[j] = bi;
      }
    }
    __syncthreads();
    const int p = sp;
    if (p != j && tid < L) {  // swap rows j and p (column tid)
      const float2 a = A[tid * LP + j];
      A[tid * LP + j] = A[tid * LP + p];
      A[tid * LP + p] = a;
    }
    __syncthreads();
    const float2 piv = A[j * LP + j];
    const float d = piv.x * piv.x + piv.y * piv.y;
    bad |= !(d > 0.f);
    const float2 ip = d > 0.f ? make_float2(piv.x / d, -piv.y / d) : make_float2(0.f, 0.f);
    if (tid < L) f[tid] = A[j * LP + tid];  // column j
    __syncthreads();
    if (tid < L) {  // row j divided by the pivot
      const float2 a = tid == j ? make_float2(1.f, 0.f) : A[tid * LP + j];
      A[tid * LP + j] = cmul(a, ip);
    }
    __syncthreads();
    for (int e = tid; e < L * L; e += blockDim.x) {
      const int i = e % L, c = e / L;
      if (i == j) continue;
      const float2 a = c == j ? make_float2(0.f, 0.f) : A[c * LP + i];
      A[c * LP + i] = csub(a, cmul(f[i], A[c * LP + j]));
    }
    __syncthreads();
  }
  for (int j = L - 1; j >= 0; --j) {
    const int p = perm[j];
    if (p != j && tid < L) {  // swap columns j and p (row tid)
      const float2 a = A[j * LP + tid];
      A[j * LP + tid] = A[p * LP + tid];
      A[p * LP + tid] = a;
    }
    __syncthreads();
  }
  for (int e = tid; e < L * L; e += blockDim.x) P[e] = A[(e / L) * LP + e % L];
  if (bad && tid == 0) info[blockIdx.x] = 1;
}

// kscale of every member set to 0 before k_tile_red_max.
__global__ void k_tile_red_zero(const int* __restrict__ ids, int cnt, float* __restrict__ sc) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < cnt; i += gridDim.x * blockDim.x) sc[ids[i]] = 0.f;
}

// Largest |W| entry of member blockIdx.y (the swept matrix at Kw + koff, side
// nl, holds -W in its lower triangle): work-group blockIdx.x covers one chunk
// of the n_t x n_t entries and folds its maximum into the member's kscale
// with an atomic max on the bits (the values are >= 0, whose order the bits
// keep).
__global__ void __launch_bounds__(256)
k_tile_red_max(const float2* __restrict__ Kw, const int* __restrict__ ncol, const unsigned short* __restrict__ cols,
               const int* __restrict__ ids, const long* __restrict__ koff, const int* __restrict__ nl, int T,
               float* __restrict__ sc) {
  const int i = blockIdx.y;
  const int tb = ids[i];
  const int nk = ncol[tb];
  const long nn = (long)nk * nk;
  const long e0 = (long)blockIdx.x * kBuildChunk;
  if (e0 >= nn) return;
  const long e1 = e0 + kBuildChunk < nn ? e0 + kBuildChunk : nn;
  const unsigned short* ct = cols + (long)tb * T * T;
  const float2* A = Kw + koff[i];
  const int n = nl[i];
  float mx = 0.f;
  for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
    const int p = (int)(e % nk), q = (int)(e / nk);
    if (p < q || ct[p] == kPadCol || ct[q] == kPadCol) continue;  // the lower triangle holds -W
    const float2 v = A[(long)q * n + p];
    mx = fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y)));
  }
  __shared__ float red[4];
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    if (m > 0.f) atomicMax(reinterpret_cast<unsigned int*>(sc + tb), __float_as_uint(m));
  }
}

// W16 of member blockIdx.y: W / scale in FP16 (W = minus the swept matrix),
// the blocks (bi, bj <= bi) of its lower triangle (kBlkW x kBlkW each, column-major, zero beyond
// n_t) in row-major block order at woff[tb]; work-group blockIdx.x covers one
// chunk.  The matrix side nl is a multiple of kBlkW (= kBlk).
__global__ void __launch_bounds__(256)
k_tile_red_pack(const float2* __restrict__ Kw, const int* __restrict__ ncol, const unsigned short* __restrict__ cols,
                const int* __restrict__ ids, const long* __restrict__ koff, const int* __restrict__ nl,
                const long* __restrict__ woff, const float* __restrict__ sc, __half2* __restrict__ W16, int T) {
  constexpr int B = kBlkW;
  const int i = blockIdx.y;
  const int tb = ids[i];
  const int nk = ncol[tb];
  const int n = nl[i];
  const int nB = n / B;
  const long total = (long)nB * (nB + 1) / 2 * B * B;
  const long e0 = (long)blockIdx.x * kBuildChunk;
  if (e0 >= total) return;
  const long e1 = e0 + kBuildChunk < total ? e0 + kBuildChunk : total;
  const unsigned short* ct = cols + (long)tb * T * T;
  const float2* A = Kw + koff[i];
  const float r = sc[tb] > 0.f ? 1.f / sc[tb] : 0.f;  // 0: W_t = 0
  __half2* Wt = W16 + woff[tb];
  for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
    const int b = (int)(e / (B * B)), w = (int)(e % (B * B));
    int bi = (int)((sqrtf(8.f * b + 1.f) - 1.f) * 0.5f);  // block row: bi (bi + 1) / 2 <= b
    while (bi * (bi + 1) / 2 > b) --bi;
    while ((bi + 1) * (bi + 2) / 2 <= b) ++bi;
    const int bj = b - bi * (bi + 1) / 2;
    const int p = bi * B + w % B, q = bj * B + w / B;
    float2 v = make_float2(0.f, 0.f);
    if (p < nk && q < nk && ct[p] != kPadCol && ct[q] != kPadCol) {
      const float2 a = p >= q ? A[(long)q * n + p] : A[(long)p * n + q];  // the sweep leaves -W, lower
      v = make_float2(-a.x * r, -a.y * r);
    }
    Wt[e] = __floats2half2_rn(v.x, v.y);
  }
}

// ---------------------------------------------------------------------------
// reduced form: application
// ---------------------------------------------------------------------------

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));

constexpr int kXsRow = kBlkW + 4;        // LDS stride of one column of inputs (bank-conflict free 16-byte reads)

// Position of row p of a block row among its inputs and products, and the row
// at a position: in every 32 rows the even ones first, as the MFMA operands of
// k_tile_ws hold them.
__device__ inline int xpos(int p) { return (p & ~31) | (p & 1) << 4 | (p & 31) >> 1; }
__device__ inline int xrow(int q) { return (q & ~31) | (q & 15) << 1 | (q >> 4 & 1); }

// The tile inputs x_t[S] of system blockIdx.y and tile blockIdx.x (io.v scaled
// by 1 / *(io.nrm + s sNrm bytes) when io.nrm is given), as the right-hand
// operand of k_tile_ws: every value is scaled by the power of two that brings
// the tile's largest component to [2^14, 2^15) and cut into kSplits FP16
// parts, x = hi + mid + lo, which hold all 24 bits of the FP32 values down to 2^-15
// of the tile's largest and resolve smaller ones to 2^-39 of it (W is stored to
// 2^-11).  Group v = s / VP of the systems, column
// n(s) = s % VP: with VP = 16 one dword (re, im) per value and column n; with
// VP = 8 the two columns 2n and 2n + 1 hold (re, -im) and (im, re).  Layout
// [group][block row][part][16 columns][kBlkW], rows at xpos().  xinv[s][tile] is the inverse
// of the scale.  Each map's tiles own xblk[map] block rows (bloc: the tile's
// first).  A few tiles and systems leave CUs idle: then `parts` work-groups
// share a tile (blockIdx.x = tile * parts + part), each finding the maximum of
// all of it and writing its share.
template <int T, int VP>
__global__ void __launch_bounds__(1024)
k_tile_xs(const int* __restrict__ ncol, const unsigned short* __restrict__ cols, const int* __restrict__ bloc,
          int maps1, int parts, FnoIO io, unsigned* __restrict__ Xs, long sXs, float* __restrict__ xinv,
          const int* __restrict__ done, long sd, int N) {
  constexpr int M2 = T * T;
  constexpr int PT = M2 / 1024;  // values per thread
  __shared__ float red[16];
  const int nt = N / T;
  const int s = blockIdx.y, t = blockIdx.x / parts, part = blockIdx.x % parts;
  // two latencies, of n and cols and of v behind them: the norm and the flag
  // are tested once those loads are in flight
  const int dn = done ? *boff(done, (long)s * sd) : 0;
  const long tb = (long)(maps1 ? 0 : s) * nt * nt + t;
  const int n = ncol[tb];
  const unsigned short* ct = cols + tb * M2;
  const float2* v = io.v + (long)s * io.sV;
  float2 xv[PT];
  int cell[PT];
#pragma unroll
  for (int k = 0; k < PT; ++k) cell[k] = ct[threadIdx.x + 1024 * k];
#pragma unroll
  for (int k = 0; k < PT; ++k) {  // padding slots load a cell too, so that no load waits behind a branch
    if ((int)threadIdx.x + 1024 * k >= n) cell[k] = kPadCol;
    xv[k] = v[tile_cell(t, cell[k] == kPadCol ? 0 : cell[k], nt, T, N)];
  }
  float sc = 1.f;
  if (io.nrm) {
    const double d = *boff(io.nrm, (long)s * io.sNrm);
    sc = d > 0.0 ? (float)(1.0 / d) : 0.f;
  }
  if (dn || n == 0) return;
  const int np = (n + kBlkW - 1) / kBlkW * kBlkW;
  float mx = 0.f;
#pragma unroll
  for (int k = 0; k < PT; ++k) {
    xv[k].x = cell[k] == kPadCol ? 0.f : xv[k].x * sc;
    xv[k].y = cell[k] == kPadCol ? 0.f : xv[k].y * sc;
    mx = fmaxf(mx, fmaxf(fabsf(xv[k].x), fabsf(xv[k].y)));
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 16; ++k) mx = fmaxf(mx, red[k]);
  // scale 2^e: the exponent is clamped so that the scale and its inverse are normal numbers
  int e = 0;
  if (mx > 0.f && mx < __builtin_huge_valf()) e = 141 - (int)(__float_as_uint(mx) >> 23);
  e = e > 126 ? 126 : (e < -126 ? -126 : e);
  const float up = __uint_as_float((unsigned)(e + 127) << 23);
  if (threadIdx.x == 0) xinv[(long)s * nt * nt + t] = __uint_as_float((unsigned)(127 - e) << 23);
  const int col = s % VP;
  unsigned* X = Xs + (long)(maps1 ? s / VP : s) * sXs + (long)bloc[tb] * kXsBlk;
#pragma unroll
  for (int k = 0; k < PT; ++k) {
    const int p = threadIdx.x + 1024 * k;
    if (p >= np) break;
    if (k % parts != part) continue;
    float re = xv[k].x * up, im = xv[k].y * up;
    unsigned* Xp = X + (long)(p / kBlkW) * kXsBlk + xpos(p % kBlkW);
#pragma unroll
    for (int q = 0; q < kSplits; ++q) {
      const _Float16 a = (_Float16)re, b = (_Float16)im;
      re -= (float)a;
      im -= (float)b;
      const unsigned ua = __builtin_bit_cast(unsigned short, a), ub = __builtin_bit_cast(unsigned short, b);
      if constexpr (VP == 16) {
        Xp[(q * 16 + col) * kBlkW] = ua | ub << 16;
      } else {
        const int cn = maps1 ? 2 * col : 0;
        Xp[(q * 16 + cn) * kBlkW] = ua | (ub ^ 0x8000u) << 16;
        Xp[(q * 16 + cn + 1) * kBlkW] = ub | ua << 16;
      }
    }
  }
}

// The products with W_t of up to VP = 8 NT systems of one map.  W_t is complex
// symmetric (W_t = (D_S^{-1} - G_SS)^{-1}, G symmetric), so only its lower
// triangle is stored, in kBlkW x kBlkW blocks.  A work-group takes a strip of
// them: block columns j0 = 2 sj and j0 + 1 of its tile (SC = 1: column j0 = sj
// alone), block rows i of [si R, si R + R) with i >= j0 (R = 1, 2, 4 or 8, by
// map), and forms for every block (i, j) B x_j (added up over the columns, per row)
// and, for j < i, B^T x_i (added up over the rows, per column): SC + R partial
// products of kBlkW values per system, which k_tile_wsum adds up.
//
// What bounds it is the stream of W (64 KB a block), which is read once.  The
// contraction runs on the matrix cores (FP16 inputs, FP32 sums): W is FP16 as
// stored, and the FP32 inputs enter as three FP16 parts (k_tile_xs), so the
// products are those of the FP32 values down to 2^-15 of a tile's largest.  Complex arithmetic is real arithmetic
// on interleaved parts: a dword (re, im) of W meets the dword (re, -im) of x
// for the real part and (im, re) for the imaginary part, 16 complex values of
// K per MFMA.
//   B x_j:    lane (a, g) of wave w loads rows 32 w + 2 a, 2 a + 1 of four
//             columns (8 bytes each, 128-byte segments); the four columns'
//             values of one row are that lane's 8 K-values of an MFMA.
//   B^T x_i:  the same registers, transposed by the matrix core: an MFMA with
//             a 0/1 right operand that picks the real (imaginary) parts leaves
//             column a's values of rows 4 g .. 4 g + 3 in lane (a, g), which
//             are then packed back to FP16 (exactly) as the left operand.  (A
//             second read of the block in the other layout cost as much as the
//             first: the blocks in flight exceed an XCD's L2.)
// Rows and columns are taken in the order of xpos().  x_j of the two columns
// stays in LDS; a wave needs x_i at its own 32 rows only, which go straight to
// registers, so the loop over the rows has no barrier.  A wave's sums of B^T x_i
// run over its own rows and are added up over the four waves at the end.  Each
// of the 16 KB that a wave needs of a block is loaded again for the next block
// as soon as it is used, D steps of 2 KB ahead; every such load is issued
// unconditionally (the last block again where there is no next), so that the
// compiler's waits know how many loads are younger than the ones waited for.
//
// KIND: strips of one row need no second set of x_i, and their last block is known
// when compiled, so nothing is loaded in vain: three work-groups per CU instead of
// two cover each other's first loads and last sums (sixteen maps at N = 128, T =
// 64: 114 us with strips of two blocks, two per CU; 96 with three; 94.6 with
// single blocks).
//
// At N = 512, T = 128 on a map of the benchmark (1.33 GB of W; a plain
// non-temporal read of as much takes 190 us): one system 225-236 us (5.8 TB/s),
// 16 systems 337 us.  The vector-ALU kernel before it, which took one block
// and one system at a time, took 272 and 3,000 us (202 us of arithmetic per
// system).  One FP16 part instead of three would save 19 us at one system.
// Two groups of 4 waves with 8 K-steps in flight took 249 us; R = 4 and 16
// (rows per strip) instead of 8 took 252 and 241 us.
template <int NT, int KIND>
__global__ void __launch_bounds__(256, KIND != kLongStrip && NT == 1 ? 3 : 2)
k_tile_ws(const unsigned* __restrict__ W16, const Strip* __restrict__ stab, const int* __restrict__ sstart,
          const int* __restrict__ scount, const int* __restrict__ ssize, int maps1, int nsys,
          const unsigned* __restrict__ Xs, long sXs, float4_t* __restrict__ Pw, long spw,
          const int* __restrict__ done, long sd) {
  constexpr int B = kBlkW, VP = 8 * NT, KS = B / 16;
  constexpr int SC = KIND == kBlockStrip ? 1 : 2;
  constexpr bool ONE = KIND != kLongStrip;          // one block row
  constexpr int D = NT == 1 ? 4 : 2;                // K-steps of W in flight (2 KB per wave each)
  constexpr int kSlot = kSplits * 16 * kXsRow;      // dwords of one block row's inputs in LDS
  static_assert(SC * kSlot * sizeof(unsigned) >= 3 * KS * 64 * sizeof(float4_t), "the waves' sums fit the inputs' LDS");
  __shared__ unsigned lds[SC * kSlot];
  const int grp = blockIdx.y, map = maps1 ? 0 : grp;
  const int size = ssize[map], R = ONE ? 1 : size & 255;
  if ((int)blockIdx.x >= scount[map] || size >> 8 != SC) return;
  const int nv = maps1 ? (nsys - grp * VP < VP ? nsys - grp * VP : VP) : 1;
  if (done) {  // uniform over the work-group
    bool all = true;
    for (int k = 0; k < nv; ++k) all &= *boff(done, (long)((maps1 ? grp * VP : grp) + k) * sd) != 0;
    if (all) return;
  }
  const Strip sp = stab[sstart[map] + blockIdx.x];
  const int nB = sp.nB, j0 = sp.j0, i0 = sp.i0, iend = i0 + R < nB ? i0 + R : nB;
  const int ibeg = i0 > j0 ? i0 : j0;
  const int tid = threadIdx.x, lane = tid & 63, a = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // in a scalar register, with all that follows from it
  const unsigned* Wt = W16 + sp.woff + 32 * w;
  const unsigned voff = (8 * g * B + 2 * a) * sizeof(unsigned);
  const unsigned* X = Xs + (long)grp * sXs + (long)sp.bloc * kXsBlk;
  const int ncols = NT == 2 ? nv : 2 * nv;  // columns in use: the others are not copied, and their sums not kept

  uint2_t A[D][4];
  const auto load_a = [&](int i, int j, int k) {  // K-step k: columns 32 (k / 2) + 8 g + 2 c + k % 2, positions 16 k + 4 g + c
    const char* Bp = reinterpret_cast<const char*>(Wt + (long)(i * (i + 1) / 2 + j) * B * B + (32 * (k >> 1) + (k & 1)) * B);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      A[k % D][c] = __builtin_nontemporal_load(reinterpret_cast<const uint2_t*>(Bp + voff + 2 * c * B * sizeof(unsigned)));
  };
  // x_i at the wave's rows, loaded a block ahead of its first use and before the loads of W that follow it; the
  // columns not in use repeat column 0 (with one system, 14 of 16: 21 of every 152 KB read)
  const int ax = a < ncols ? a : 0;
  uint4_t xr[2][kSplits], xn[2][kSplits];
  const auto load_x = [&](int i, uint4_t (*to)[kSplits]) {
    const unsigned* xi = X + (long)i * kXsBlk + 32 * w + ax * B + 4 * g;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < kSplits; ++q) to[h][q] = *reinterpret_cast<const uint4_t*>(xi + q * 16 * B + 16 * h);
  };
  load_x(ibeg == j0 && ibeg + 1 < iend ? ibeg + 1 : ibeg, xr);
#pragma unroll
  for (int k = 0; k < D; ++k) load_a(ibeg, j0, k);

  {  // x_j of the two columns, the columns in use, into LDS
    const unsigned* src = X + (long)j0 * kXsBlk;
    const int per = ncols * (B / 4), all = (SC == 2 && j0 + 1 < nB ? 2 : 1) * kSplits * per;
    for (int e0 = tid; e0 < all; e0 += 4 * 256) {
      uint4_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = e0 + u * 256 < all ? e0 + u * 256 : tid, q = e / per, r = (e - q * per) >> 5, c = e & 31;
        v[u] = *reinterpret_cast<const uint4_t*>(src + (q * 16 + r) * B + 4 * c);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = e0 + u * 256, q = e / per, r = (e - q * per) >> 5, c = e & 31;
        if (e < all) *reinterpret_cast<uint4_t*>(lds + (q * 16 + r) * kXsRow + 4 * c) = v[u];
      }
    }
  }
  // the 0/1 operands: value 4 g + c of the K-step to column a, real or imaginary part
  half8_t Ire, Iim;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const _Float16 one = (_Float16)(4 * g + c == a ? 1.f : 0.f);
    Ire[2 * c] = one;
    Ire[2 * c + 1] = (_Float16)0.f;
    Iim[2 * c] = (_Float16)0.f;
    Iim[2 * c + 1] = one;
  }
  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  float4_t Z[SC][KS][NT];
#pragma unroll
  for (int h = 0; h < SC; ++h)
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int n = 0; n < NT; ++n) Z[h][k][n] = zero;

  // partial products: [strip][SC columns, R rows][positions / 4][system][re, im] float4
  const long qlen = 64 * nv;
  float4_t* P = Pw + (long)grp * spw + (long)blockIdx.x * (SC + R) * qlen;
  const auto put_p = [&](float4_t* Pq, int k, const float4_t* acc) {  // positions 16 k + 4 g .. + 3
    float4_t* q = Pq + (k * 4 + g) * 2 * nv;
    if constexpr (NT == 2) {
      if (a < nv) {
        q[2 * a] = acc[0];
        q[2 * a + 1] = acc[1];
      }
    } else {
      if (a < 2 * nv) q[a] = acc[0];
    }
  };
  const auto mac = [&](half8_t h, uint4_t v, float4_t* acc) {
    if constexpr (NT == 2) {
      const half8_t re = __builtin_bit_cast(half8_t, v ^ 0x80000000u);
      const half8_t im = __builtin_bit_cast(half8_t, (v >> 16) | (v << 16));
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h, re, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h, im, acc[1], 0, 0, 0);
    } else {
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h, __builtin_bit_cast(half8_t, v), acc[0], 0, 0, 0);
    }
  };
  float4_t Y[2 * NT];
  // block (i, j): its row sums to Y, with `columns` its column sums to Zj (not on the diagonal, where the block is
  // whole and its row sums are all), and the loads of block (ni, nj), unless it is the `last`
  const auto product = [&](auto columns, auto last, int i, int j, int ni, int nj, const unsigned* xj,
                           float4_t (&Zj)[KS][NT]) {
    int xoff = a * kXsRow + 4 * g;
    asm volatile("" : "+v"(xoff));  // x_j is read from LDS for every block: 96 registers otherwise
    unsigned keep = i != j ? 0xFFFFFFFFu : 0u;
    asm volatile("" : "+v"(keep));  // masked, not branched around: see load_a
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      half8_t f[2];
      {
        const uint2_t* Ak = A[k % D];
        f[0] = __builtin_bit_cast(half8_t, (uint4_t{Ak[0].x, Ak[1].x, Ak[2].x, Ak[3].x}));
        f[1] = __builtin_bit_cast(half8_t, (uint4_t{Ak[0].y, Ak[1].y, Ak[2].y, Ak[3].y}));
      }
      if (k + D < KS) load_a(i, j, k + D);
      else if constexpr (!decltype(last)::value) load_a(ni, nj, k + D - KS);
#pragma unroll
      for (int q = 0; q < kSplits; ++q) {
        const uint4_t v = *reinterpret_cast<const uint4_t*>(xj + xoff + q * 16 * kXsRow + 16 * k);
        mac(f[0], v, Y);
        mac(f[1], v, Y + NT);
      }
      if constexpr (decltype(columns)::value) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float4_t re = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[h], Ire, zero, 0, 0, 0);
          const float4_t im = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[h], Iim, zero, 0, 0, 0);
          uint4_t tr;
#pragma unroll
          for (int c = 0; c < 4; ++c) tr[c] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(re[c], im[c])) & keep;
          const half8_t ft = __builtin_bit_cast(half8_t, tr);
#pragma unroll
          for (int q = 0; q < kSplits; ++q) mac(ft, xr[h][q], Zj[k]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of their use
    }
  };
  const auto store_y = [&](int i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) put_p(P + (SC + i - i0) * qlen, 2 * w + h, Y + h * NT);
  };
  __syncthreads();
  typedef std::true_type yes;
  typedef std::false_type no;
  int i = ibeg;
  if (i == j0) {
#pragma unroll
    for (int k = 0; k < 2 * NT; ++k) Y[k] = zero;
    const bool more = i + 1 < iend;
    product(no(), std::integral_constant<bool, ONE>(), i, j0, more ? i + 1 : i, j0, lds, Z[0]);
    store_y(i);
    ++i;
  }
  if constexpr (ONE) {
    if (i < iend) {
#pragma unroll
      for (int k = 0; k < 2 * NT; ++k) Y[k] = zero;
      product(yes(), std::integral_constant<bool, SC == 1>(), i, j0, i, j0 + 1, lds, Z[0]);
      if constexpr (SC == 2) product(yes(), yes(), i, j0 + 1, i, j0 + 1, lds + kSlot, Z[SC - 1]);
      store_y(i);
    }
  } else {
    for (; i < iend; ++i) {
      const bool more = i + 1 < iend;
#pragma unroll
      for (int k = 0; k < 2 * NT; ++k) Y[k] = zero;
      product(yes(), no(), i, j0, i, j0 + 1, lds, Z[0]);
      if constexpr (NT == 1) load_x(more ? i + 1 : i, xn);
      product(yes(), no(), i, j0 + 1, more ? i + 1 : i, more ? j0 : j0 + 1, lds + kSlot, Z[SC - 1]);
      store_y(i);
      if constexpr (NT == 1) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < kSplits; ++q) xr[h][q] = xn[h][q];
      } else {
        load_x(more ? i + 1 : i, xr);
      }
    }
  }
  // Z over the four waves: wave w keeps positions 32 w .. 32 w + 31
  float4_t* red = reinterpret_cast<float4_t*>(lds);
#pragma unroll
  for (int h = 0; h < SC; ++h) {
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if ((k >> 1) != w) red[((w - (w > (k >> 1))) * KS + k) * 64 + lane] = Z[h][k][n];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if ((k >> 1) == w) Z[h][k][n] += (red[k * 64 + lane] + red[(KS + k) * 64 + lane]) + red[(2 * KS + k) * 64 + lane];
    }
    if (j0 + h < nB)
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if ((k >> 1) == w) put_p(P + h * qlen, k, Z[h][k]);
  }
}

// u_t of block row blockIdx.x % nbmax of tile blockIdx.x / nbmax, systems of
// group blockIdx.z, 64 of the 64 nv values (float4: four rows) a system group
// has per block row: the partial products of the strips of the row and
// of the column, in four interleaved sums (one per slice of 64 threads, each in
// a fixed order) added up in LDS, times the tile's scales, written to U at the
// cells of S.
template <int T, int VP>
__global__ void __launch_bounds__(256)
k_tile_wsum(const float* __restrict__ ksc, const float* __restrict__ xinv, const int* __restrict__ ncol,
            const unsigned short* __restrict__ cols, const int* __restrict__ sloc, const int* __restrict__ spos,
            const int* __restrict__ ssize, int maps1, int nsys, int nbmax, const float4_t* __restrict__ Pw, long spw,
            float2* __restrict__ U, const int* __restrict__ done, long sd, int N) {
  constexpr int M2 = T * T, B = kBlkW;
  __shared__ float4_t red[4][64];
  const int nt = N / T;
  const int grp = blockIdx.z, map = maps1 ? 0 : grp;
  const int nv = maps1 ? (nsys - grp * VP < VP ? nsys - grp * VP : VP) : 1;
  if ((int)blockIdx.y >= nv) return;
  const int t = blockIdx.x / nbmax, i = blockIdx.x % nbmax;
  const long tb = (long)map * nt * nt + t;
  const int n = ncol[tb], nB = (n + B - 1) / B;
  if (i >= nB) return;
  const int R = ssize[map] & 255, SC = ssize[map] >> 8, si = i / R, sj = SC == 2 ? i >> 1 : i;
  const int nS = (nB + R - 1) / R;
  const int e = threadIdx.x & 63, sl = threadIdx.x >> 6;
  const long qlen = 64 * nv;
  const float4_t* P = Pw + (long)grp * spw + 64 * blockIdx.y + e;
  const int* pos = spos + sloc[tb];  // place of each of the tile's strips in the map's list, [si][64]
  float4_t acc = {0.f, 0.f, 0.f, 0.f};
  // terms 0 .. sj: row sums of strips (si, 0 .. sj); then column sums of (si .. nS - 1, sj)
  const int terms = sj + 1 + nS - si;
#pragma unroll 4
  for (int k = sl; k < terms; k += 4) {
    const int r = k <= sj ? si : si + k - sj - 1, c = k <= sj ? k : sj;
    acc += P[((long)pos[r * 64 + c] * (SC + R) + (k <= sj ? SC + i - si * R : i & (SC - 1))) * qlen];
  }
  red[sl][e] = acc;
  __syncthreads();
  if (threadIdx.x >= 32) return;
  const int e2 = 32 * blockIdx.y + threadIdx.x;
  const int v = e2 % nv, h = e2 / nv;
  const int pos0 = 4 * h;  // its first position in the block row
  const int s = (maps1 ? grp * VP : grp) + v;
  if (done && *boff(done, (long)s * sd)) return;
  const int f = 2 * threadIdx.x;
  const float4_t re = (red[0][f] + red[1][f]) + (red[2][f] + red[3][f]);
  const float4_t im = (red[0][f + 1] + red[1][f + 1]) + (red[2][f + 1] + red[3][f + 1]);
  const float k1 = ksc[tb], k2 = xinv[(long)s * nt * nt + t];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int p = i * B + xrow(pos0 + r);
    if (p < n) {
      const int c = cols[tb * M2 + p];
      if (c != kPadCol) U[((long)s * nt * nt + t) * M2 + c] = make_float2(re[r] * k1 * k2, im[r] * k1 * k2);
    }
  }
}

// Last pass of the tile convolution and the application's result, z = x + G_t
// u_t: the inverse row transforms of k_pass3 (rows of tile blockIdx.y % tiles,
// system blockIdx.y / tiles), whose rows are then read and written in the
// grid's order; x is io.v scaled as in k_tile_xs and is written to io.vw when
// io.nrm and io.vw are given.  Bound by memory: T x 2T transformed values in, x
// in, z out; a kernel of its own for the sum read and wrote T x T more, 21 of
// 523 us for 16 systems at N = 512, T = 128, and its launch 2 of 33 us for one
// system at N = 128, T = 64.
template <int T>
struct TileOut {
  static constexpr int M = 2 * T, E = kFftE<M>, NT = FftShape<M, E>::NT, ROWS = 256 / NT;
};
template <int T>
__global__ void __launch_bounds__(256)
k_tile_out(FnoIO io, const float2* __restrict__ Tm, const float2* __restrict__ tw, const int* __restrict__ done,
           long sd, int N) {
  typedef TileOut<T> S;
  constexpr int M = S::M, E = S::E, NT = S::NT;
  __shared__ __align__(16) float2 smem[S::ROWS * LdsLen<M>::value];
  const int nt = N / T;
  const int s = blockIdx.y / (nt * nt), tile = blockIdx.y % (nt * nt);
  const int dn = done ? *boff(done, (long)s * sd) : 0;  // tested once the loads are in flight
  const int t = threadIdx.x % NT, rl = threadIdx.x / NT, row = blockIdx.x * S::ROWS + rl;
  Tm += (long)blockIdx.y * T * M;
  FftTwiddles<float, M, E> tws;
  tws.load(tw, t);
  float2 v[E], xv[E / 2];
#pragma unroll
  for (int k = 0; k < E; ++k) v[k] = Tm[tpos(row, t + k * NT, T)];
  const long cell = (long)(tile / nt * T + row) * N + tile % nt * T;
#pragma unroll
  for (int k = 0; k < E / 2; ++k) xv[k] = io.v[(long)s * io.sV + cell + t + k * NT];
  float sc = 1.f;
  if (io.nrm) {
    const double d = *boff(io.nrm, (long)s * io.sNrm);
    sc = d > 0.0 ? (float)(1.0 / d) : 0.f;
  }
  if (dn) return;
  reg_fft<float, M, +1, false, true, E>(v, smem + rl * LdsLen<M>::value, tws, t);  // columns < T are used
  constexpr float inv = 1.f / ((float)M * (float)M);
#pragma unroll
  for (int k = 0; k < E / 2; ++k) {
    const long e = cell + t + k * NT;
    float2 x = xv[k];
    x.x *= sc;
    x.y *= sc;
    if (io.nrm && io.vw) io.vw[(long)s * io.sV + e] = x;
    io.z[(long)s * io.sZ + e] = cadd(x, cscale(v[k], inv));
  }
}

// Inputs and partial products of the applications to up to nsys systems.
// One map serves groups of 8 or 16 systems; systems with maps of their own
// are groups of one.
int grow_products(cgm_tiles* t, int nsys) {
  const size_t sys = (size_t)std::max(nsys, 1);
  const size_t groups = t->maps1 ? (sys + 15) / 16 : sys, per = t->maps1 ? std::min<size_t>(sys, 16) : 1;
  int rc = grow(t, &t->Pw, &t->pw_cap, groups * t->plen_max * 64 * per);
  if (!rc) rc = grow(t, &t->Xs, &t->xs_cap, groups * t->xblk_max * kXsBlk);
  if (!rc) rc = grow(t, &t->xinv, &t->xinv_cap, sys * t->nt * t->nt);
  return rc;
}

void release_scratch(cgm_tiles* t) {
  void* ptrs[] = {t->U, t->Tm};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  t->U = t->Tm = nullptr;
  const size_t n = (size_t)t->N * t->N, tm = (size_t)t->nt * t->nt * t->T * t->P.M;
  t->bytes -= (n + tm) * sizeof(float2) * t->scratch_sys;
  t->scratch_sys = 0;
}

// The apply scratch for nsys systems; where one of its buffers cannot be had,
// none counts (scratch_sys = 0) and the next application asks for all again.
int ensure_scratch(cgm_tiles* t, int nsys) {
  if (nsys <= t->scratch_sys) return CGM_SUCCESS;
  release_scratch(t);
  const size_t n = (size_t)t->N * t->N;
  const size_t tm = (size_t)t->nt * t->nt * t->T * t->P.M;
  int rc = CGM_SUCCESS;
  if (hipMalloc((void**)&t->U, sizeof(float2) * n * nsys) != hipSuccess ||
      hipMalloc((void**)&t->Tm, sizeof(float2) * tm * nsys) != hipSuccess) {
    (void)hipGetLastError();
    cgm_set_last_error("tile preconditioner: scratch allocation for %d systems failed", nsys);
    rc = CGM_ERROR_ALLOC;
  }
  // the cells with chi = 0 keep u = 0: the application writes only the cells of
  // S, on a stream that need not wait for the null stream's clear
  if (!rc && (hipMemset(t->U, 0, sizeof(float2) * n * nsys) != hipSuccess ||
              hipStreamSynchronize(nullptr) != hipSuccess)) {
    cgm_set_last_error("tile preconditioner: scratch clear failed");
    rc = CGM_ERROR_DEVICE;
  }
  if (!rc) rc = grow_products(t, nsys);
  if (rc) {
    release_scratch(t);
    return rc;
  }
  t->scratch_sys = nsys;
  t->bytes += (n + tm) * sizeof(float2) * nsys;
  return CGM_SUCCESS;
}

// u_t = W_t x_t[S] of every tile for nsys systems; NT = 1: groups of up to 8
// systems of one map (or one system with its own map), NT = 2: up to 16.  Each
// column of the MFMAs is one system's, so a system's result does not depend on
// the others or on NT.
template <int T, int NT>
int launch_ws(const cgm_tiles* tl, hipStream_t st, const FnoIO& io, const int* done, long sd, int nsys,
              hipEvent_t* ev) {
  constexpr int VP = 8 * NT;
  const int ntiles = tl->nt * tl->nt;
  const int m1 = tl->maps1 ? 1 : 0;
  const int groups = m1 ? (nsys + VP - 1) / VP : nsys;
  const int per = m1 ? std::min(nsys, VP) : 1;
  const int parts = ntiles * nsys < 128 ? 4 : 1;
  const long spw = tl->plen_max * 64 * per, sxs = (long)tl->xblk_max * kXsBlk;
  float4_t* Pw = reinterpret_cast<float4_t*>(tl->Pw);
  hipLaunchKernelGGL((k_tile_xs<T, VP>), dim3(ntiles * parts, nsys), dim3(1024), 0, st, tl->ncol, tl->cols, tl->bloc, m1, parts, io,
                     tl->Xs, sxs, tl->xinv, done, sd, tl->N);
  if (ev) CGM_HIP(hipEventRecord(ev[0], st));
  const auto ws = [&](auto kind) {
    hipLaunchKernelGGL((k_tile_ws<NT, decltype(kind)::value>), dim3(tl->scount_max, groups), dim3(256), 0, st,
                       reinterpret_cast<const unsigned*>(tl->W16), tl->stab, tl->sstart, tl->scount, tl->ssize, m1,
                       nsys, tl->Xs, sxs, Pw, spw, done, sd);
  };
  // single rows have a launch of their own only where no map has longer strips
  // (a second launch costs more than it gives: three maps at N = 192, T = 64,
  // 68 us with it and 63.7 without)
  if (tl->kinds & 1u << kLongStrip) ws(std::integral_constant<int, kLongStrip>());
  else if (tl->kinds & 1u << kRowStrip) ws(std::integral_constant<int, kRowStrip>());
  if (tl->kinds & 1u << kBlockStrip) ws(std::integral_constant<int, kBlockStrip>());
  if (ev) CGM_HIP(hipEventRecord(ev[1], st));
  hipLaunchKernelGGL((k_tile_wsum<T, VP>), dim3(ntiles * tl->nbmax, per, groups), dim3(256), 0, st, tl->kscale,
                     tl->xinv, tl->ncol, tl->cols, tl->sloc, tl->spos, tl->ssize, m1, nsys, tl->nbmax, Pw, spw, tl->U,
                     done, sd, tl->N);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

// ev, when given: events recorded around k_tile_ws (live timing).
int launch_apply_red(const cgm_tiles* tl, hipStream_t st, const FnoIO& io, const int* done, long sd, int nsys,
                     hipEvent_t* ev) {
  cgm_tiles* t = const_cast<cgm_tiles*>(tl);  // the apply scratch grows with the batch
  int rc = ensure_scratch(t, nsys);
  if (rc) return rc;
  const int ntiles = tl->nt * tl->nt;
  const int B = nsys * ntiles;
  if (B > 65535) {
    cgm_set_last_error("%d systems exceed the tile convolution's batch limit", nsys);
    return CGM_ERROR_UNSUPPORTED;
  }
  if (tl->scount_max > 0) {
    if (tl->T == 64) {
      rc = tl->maps1 && nsys > 8 ? launch_ws<64, 2>(tl, st, io, done, sd, nsys, ev)
                                 : launch_ws<64, 1>(tl, st, io, done, sd, nsys, ev);
    } else {
      rc = tl->maps1 && nsys > 8 ? launch_ws<128, 2>(tl, st, io, done, sd, nsys, ev)
                                 : launch_ws<128, 1>(tl, st, io, done, sd, nsys, ev);
    }
    if (rc) return rc;
  } else if (ev) {  // no cell of chi != 0: nothing streamed
    CGM_HIP(hipEventRecord(ev[0], st));
    CGM_HIP(hipEventRecord(ev[1], st));
  }
  BatchStrides bs;
  bs.x = tl->M2;
  bs.y = tl->M2;
  bs.T = (long)tl->T * tl->P.M;
  rc = launch_pass1<float>(tl->P, st, tl->U, nullptr, nullptr, nullptr, kModeGreen, tl->Tm, tl->tw32, nullptr, B, bs);
  if (!rc) rc = launch_pass2<float, float2>(tl->P, st, tl->Tm, tl->gq, tl->tw32, nullptr, B, bs);
  if (rc) {
    cgm_set_last_error("tile convolution at T = %d failed", tl->T);
    return rc;
  }
  if (tl->T == 64)
    hipLaunchKernelGGL((k_tile_out<64>), dim3(64 / TileOut<64>::ROWS, B), dim3(256), 0, st, io, tl->Tm, tl->tw32,
                       done, sd, tl->N);
  else
    hipLaunchKernelGGL((k_tile_out<128>), dim3(128 / TileOut<128>::ROWS, B), dim3(256), 0, st, io, tl->Tm, tl->tw32,
                       done, sd, tl->N);
  CGM_HIP(hipGetLastError());
  return CGM_SUCCESS;
}

// The storage of W of maps 0 .. maps-1 from n_t (nc, [maps][tiles]): block
// lists, offsets, entries streamed per map; uploads them and sizes W16 and the
// partial products.
int layout_reduced(cgm_tiles* t, const std::vector<int>& nc, int maps) {
  hipStream_t st = t->ctx->stream;
  const int ntiles = t->nt * t->nt;
  const int nb = ntiles * maps;
  constexpr long BB = (long)kBlkW * kBlkW;
  std::vector<long> off(nb);
  std::vector<int> bloc(nb), sloc(nb), spos, sstart(maps), scount(maps), ssize(maps);
  std::vector<Strip> stab;
  long total = 0;
  t->kept.assign(maps, 0.0);
  t->nbmax = t->scount_max = t->xblk_max = 0;
  t->plen_max = 0;
  t->kinds = 0;
  t->maps1 = maps == 1;
  const auto blocks = [&](int m, int tl) { return (nc[m * ntiles + tl] + kBlkW - 1) / kBlkW; };
  struct Item { int work, tile, i, j; };
  // map m in strips of R block rows and C block columns
  const auto strips = [&](int m, int R, int C) {
    std::vector<Item> items;
    for (int tl = 0; tl < ntiles; ++tl) {
      const int nB = blocks(m, tl);
      for (int i = 0; i * R < nB; ++i)
        for (int j = 0; C * j < std::min(nB, i * R + R); ++j) {
          int work = 0;
          for (int r = i * R; r < std::min(nB, i * R + R); ++r) work += std::max(0, std::min(C, r - C * j + 1));
          items.push_back({work, tl, i, j});
        }
    }
    return items;
  };
  for (int m = 0; m < maps; ++m) {
    int rows = 0;
    for (int tl = 0; tl < ntiles; ++tl) {
      const int k = m * ntiles + tl;
      const int nB = blocks(m, tl);
      const int nblk = nB * (nB + 1) / 2;
      off[k] = total;
      total += nblk * BB;
      t->kept[m] += (double)nblk * BB;
      bloc[k] = rows;
      rows += nB;
      t->nbmax = std::max(t->nbmax, nB);
    }
    // long strips move fewer partial products and short ones keep more
    // work-groups busy: the longest of which each CU gets four or more; single
    // rows where two leave CUs idle (16 tiles of side 64, 336 strips of two: 52.1 us,
    // of one 54.5), and single blocks where those do (four tiles, 168 strips of
    // one row, sixteen systems: 43.2 us, single blocks 40.6; one tile, nine systems:
    // 33.2 and 28.7).  The map alone decides, so that its rounding does not depend
    // on the others.
    int R = 8, C = 2;
    std::vector<Item> items = strips(m, R, C);
    while (R > 1 && items.size() < (R == 2 ? 256 : 1024)) items = strips(m, R /= 2, C);
    if (R == 1 && items.size() < 256) items = strips(m, R, C = 1);
    ssize[m] = R | C << 8;
    if (!items.empty()) t->kinds |= 1u << (R > 1 ? kLongStrip : C == 2 ? kRowStrip : kBlockStrip);
    const int spos0 = (int)spos.size();
    int slots = 0;
    for (int tl = 0; tl < ntiles; ++tl) {
      sloc[m * ntiles + tl] = spos0 + slots;
      slots += (blocks(m, tl) + R - 1) / R * 64;
    }
    spos.resize(spos0 + slots);
    std::stable_sort(items.begin(), items.end(), [](const Item& x, const Item& y) { return x.work > y.work; });
    sstart[m] = (int)stab.size();
    for (size_t k = 0; k < items.size(); ++k) {
      const int q = m * ntiles + items[k].tile;
      spos[sloc[q] + items[k].i * 64 + items[k].j] = (int)k;
      stab.push_back({off[q], bloc[q], blocks(m, items[k].tile), items[k].i * R, items[k].j * C});
    }
    scount[m] = (int)items.size();
    t->scount_max = std::max(t->scount_max, scount[m]);
    t->plen_max = std::max(t->plen_max, (long)scount[m] * (C + R));
    t->xblk_max = std::max(t->xblk_max, rows);
  }
  int rc;
  if ((rc = grow(t, &t->W16, &t->w16_cap, (size_t)std::max(total, 1L)))) return rc;
  if ((rc = grow(t, &t->stab, &t->stab_cap, std::max<size_t>(stab.size(), 1)))) return rc;
  if ((rc = grow(t, &t->spos, &t->spos_cap, std::max<size_t>(spos.size(), 1)))) return rc;
  if ((rc = grow_products(t, t->scratch_sys))) return rc;
  CGM_HIP(hipMemcpyAsync(t->woff, off.data(), sizeof(long) * nb, hipMemcpyHostToDevice, st));
  CGM_HIP(hipMemcpyAsync(t->bloc, bloc.data(), sizeof(int) * nb, hipMemcpyHostToDevice, st));
  CGM_HIP(hipMemcpyAsync(t->sloc, sloc.data(), sizeof(int) * nb, hipMemcpyHostToDevice, st));
  if (!stab.empty()) {
    CGM_HIP(hipMemcpyAsync(t->stab, stab.data(), sizeof(Strip) * stab.size(), hipMemcpyHostToDevice, st));
    CGM_HIP(hipMemcpyAsync(t->spos, spos.data(), sizeof(int) * spos.size(), hipMemcpyHostToDevice, st));
  }
  CGM_HIP(hipMemcpyAsync(t->sstart, sstart.data(), sizeof(int) * maps, hipMemcpyHostToDevice, st));
  CGM_HIP(hipMemcpyAsync(t->scount, scount.data(), sizeof(int) * maps, hipMemcpyHostToDevice, st));
  CGM_HIP(hipMemcpyAsync(t->ssize, ssize.data(), sizeof(int) * maps, hipMemcpyHostToDevice, st));
  CGM_HIP(hipStreamSynchronize(st));  // the host vectors are read by the copies above
  return CGM_SUCCESS;
}

int upload_twiddles(cgm_tiles* t) {
  const int M = t->P.M;
  std::vector<float2> t32(M);
  std::vector<double2> t64(M);
  for (int q = 0; q < M; ++q) {
    const double a = -2.0 * CGM_PI * (double)q / (double)M;
    t64[q] = make_double2(cos(a), sin(a));
    t32[q] = make_float2((float)t64[q].x, (float)t64[q].y);
  }
  CGM_HIP(hipMemcpy(t->tw32, t32.data(), sizeof(float2) * M, hipMemcpyHostToDevice));
  CGM_HIP(hipMemcpy(t->tw64, t64.data(), sizeof(double2) * M, hipMemcpyHostToDevice));
  return CGM_SUCCESS;
}

// Symmetric block sweep (Gauss-Jordan on a symmetric matrix), in place, of
// the members' matrices A = D_S^{-1} - G_SS (side nl, column-major at
// Kw + koff, only the lower triangle kept): for every block column k0
// (kBlk wide) the pivot block is inverted (k_gj_inv, batched over the members
// still that large), then with P = A_kk^{-1} and C the block column k0 of the
// symmetric matrix,
//     A -= (C P) C^T (lower triangle, rocBLAS csyrkx);  A[:, k0 cols] = C P
//     (rows outside the pivot; the rows above land in the block row);  A_kk = -P.
// The matrix stays symmetric at every step (the sweep operator), and after
// the last block it holds -A^{-1} = -W.  No pivoting between blocks: the pivot
// blocks are Schur complements of the tile operator's restrictions to groups
// of cells, which the near-resonant but physical operators keep invertible (a
// zero pivot is reported per member).  In complex64 on the 128 x 128 tiles of
// the benchmark maps the result is within 3.5e-5 - 5.5e-5 of a complex128
// inverse (the unsymmetric block Gauss-Jordan: 3e-5 - 7e-5; LU with partial
// pivoting: 1e-5 - 2e-5), far below the FP16 storage of W, for half the
// flops of the unsymmetric form.
// Frees the FP32 matrices and blocks of the symmetric block sweep.
void release_factor_workspace(cgm_tiles* t) {
  float2** bufs[] = {&t->Kw, &t->Pb, &t->Rw, &t->Cw};
  size_t* caps[] = {&t->kw_cap, &t->pb_cap, &t->rw_cap, &t->cw_cap};
  for (int i = 0; i < 4; ++i) {
    if (*bufs[i]) (void)hipFree(*bufs[i]);
    t->bytes -= *caps[i] * sizeof(float2);
    *bufs[i] = nullptr;
    *caps[i] = 0;
  }
}

// *bad: the first member with a zero pivot, or -1.
int gj_invert(cgm_tiles* t, int members, const std::vector<int>& nlh, const std::vector<long>& koffh, int* bad) {
  hipStream_t st = t->ctx->stream;
  const int nmx = nlh[0];  // members are sorted by size, largest first
  int rc;
  if ((rc = grow(t, &t->Pb, &t->pb_cap, (size_t)members * kBlk * kBlk))) return rc;
  if ((rc = grow(t, &t->Rw, &t->rw_cap, (size_t)kBlk * nmx))) return rc;
  if ((rc = grow(t, &t->Cw, &t->cw_cap, (size_t)kBlk * nmx))) return rc;
  CGM_HIP(hipMemsetAsync(t->info, 0, sizeof(int) * members, st));
  const rocblas_float_complex one{1.f, 0.f}, mone{-1.f, 0.f}, zero{0.f, 0.f};
  const rocblas_operation nn = rocblas_operation_none;
  for (int k0 = 0; k0 < nmx; k0 += kBlk) {
    int cnt = 0;
    while (cnt < members && nlh[cnt] > k0) ++cnt;
    hipLaunchKernelGGL(k_gj_gather, dim3(cnt), dim3(256), 0, st, t->Kw, t->koff, t->nl, k0, t->Pb);
    hipLaunchKernelGGL(k_gj_inv, dim3(cnt), dim3(1024), 0, st, t->Pb, t->info);
    CGM_HIP(hipGetLastError());
    for (int i = 0; i < cnt; ++i) {
      const int n = nlh[i];
      float2* M = t->Kw + koffh[i];
      float2* P = t->Pb + (long)i * kBlk * kBlk;
      const dim3 tiles32(n / 32, kBlk / 32);
      hipLaunchKernelGGL(k_sw_gather, tiles32, dim3(256), 0, st, M, n, k0, t->Cw);
      CGM_HIP(hipGetLastError());
      rocblas_float_complex* Mr = reinterpret_cast<rocblas_float_complex*>(M);
      rocblas_float_complex* Pr = reinterpret_cast<rocblas_float_complex*>(P);
      rocblas_float_complex* C = reinterpret_cast<rocblas_float_complex*>(t->Cw);
      rocblas_float_complex* CP = reinterpret_cast<rocblas_float_complex*>(t->Rw);
      rocblas_status s = rocblas_cgemm(t->h, nn, nn, n, kBlk, kBlk, &one, C, n, Pr, kBlk, &zero, CP, n);
      if (s == rocblas_status_success)  // lower triangle of M -= (C P) C^T
        s = rocblas_csyrkx(t->h, rocblas_fill_lower, nn, n, kBlk, &mone, CP, n, C, n, &one, Mr, n);
      CGM_CHECK(s == rocblas_status_success, CGM_ERROR_DEVICE, "rocblas cgemm / csyrkx: status %d", (int)s);
      hipLaunchKernelGGL(k_sw_scatter, tiles32, dim3(256), 0, st, M, n, k0, t->Rw, P);
      CGM_HIP(hipGetLastError());
    }
  }
  std::vector<int> info(members);
  CGM_HIP(hipMemcpyAsync(info.data(), t->info, sizeof(int) * members, hipMemcpyDeviceToHost, st));
  CGM_HIP(hipStreamSynchronize(st));
  *bad = -1;
  for (int i = 0; i < members && *bad < 0; ++i)
    if (info[i]) *bad = i;
  return CGM_SUCCESS;
}

int factor_reduced(cgm_tiles* t, const double2* blk, const float* chi, long chi_stride, int maps) {
  cgm_context* c = t->ctx;
  hipStream_t st = c->stream;
  const int ntiles = t->nt * t->nt;
  const int nb = ntiles * maps;
  const int T = t->T, N = t->N;
  // spectrum of the tile convolution from the T x T corner of the block
  CGM_HIP(hipMemcpy2DAsync(t->blkT, sizeof(double2) * T, blk, sizeof(double2) * N, sizeof(double2) * T, T,
                           hipMemcpyDeviceToDevice, st));
  int rc = spectrum_from_block(t->P, st, t->blkT, t->tw64, t->gq, nullptr);
  if (rc) return rc;
  if (T == 64)
    hipLaunchKernelGGL((k_tile_cols<64>), dim3(ntiles, maps), dim3(1024), 0, st, chi, chi_stride, N, t->ncol,
                       t->cols);
  else
    hipLaunchKernelGGL((k_tile_cols<128>), dim3(ntiles, maps), dim3(1024), 0, st, chi, chi_stride, N, t->ncol,
                       t->cols);
  CGM_HIP(hipGetLastError());
  std::vector<int> nc(nb);
  CGM_HIP(hipMemcpyAsync(nc.data(), t->ncol, sizeof(int) * nb, hipMemcpyDeviceToHost, st));
  CGM_HIP(hipStreamSynchronize(st));
  // the storage of W and the factor members (tiles with n_t > 0, largest first)
  if ((rc = layout_reduced(t, nc, maps))) return rc;
  std::vector<int> mem;
  for (int k = 0; k < nb; ++k)
    if (nc[k] > 0) mem.push_back(k);
  std::stable_sort(mem.begin(), mem.end(), [&](int x, int y) { return nc[x] > nc[y]; });
  const int members = (int)mem.size();
  // u = 0 on the cells with chi = 0 of the new maps: the application writes only the cells of S
  CGM_HIP(hipMemsetAsync(t->U, 0, sizeof(float2) * (size_t)N * N * t->scratch_sys, st));
  if (members == 0) {
    CGM_HIP(hipStreamSynchronize(st));
    return CGM_SUCCESS;
  }
  std::vector<int> nlh(members);
  std::vector<long> koffh(members);
  long ktot = 0;
  int chunks = 1;
  for (int i = 0; i < members; ++i) {
    nlh[i] = (nc[mem[i]] + kBlk - 1) / kBlk * kBlk;
    koffh[i] = ktot;
    ktot += (long)nlh[i] * nlh[i];
    chunks = std::max(chunks, (int)(((long)nlh[i] * nlh[i] + kBuildChunk - 1) / kBuildChunk));
  }
  if ((rc = grow(t, &t->Kw, &t->kw_cap, (size_t)ktot))) return rc;
  CGM_HIP(hipMemcpyAsync(t->ids, mem.data(), sizeof(int) * members, hipMemcpyHostToDevice, st));
  CGM_HIP(hipMemcpyAsync(t->nl, nlh.data(), sizeof(int) * members, hipMemcpyHostToDevice, st));
  CGM_HIP(hipMemcpyAsync(t->koff, koffh.data(), sizeof(long) * members, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_tile_build_red, dim3(chunks, members), dim3(256), 0, st, blk, chi, chi_stride, t->ncol, t->cols,
                     t->ids, t->koff, t->nl, t->Kw, N, T);
  CGM_HIP(hipGetLastError());
  int bad = -1;
  if ((rc = gj_invert(t, members, nlh, koffh, &bad))) return rc;
  if (bad >= 0) {
    const int tb = mem[bad];
    cgm_set_last_error("tile %d of map %d: a pivot block of its reduced operator is singular", tb % ntiles,
                       tb / ntiles);
    return CGM_ERROR_NONFINITE;
  }
  hipLaunchKernelGGL(k_tile_red_zero, dim3(1), dim3(256), 0, st, t->ids, members, t->kscale);
  hipLaunchKernelGGL(k_tile_red_max, dim3(chunks, members), dim3(256), 0, st, t->Kw, t->ncol, t->cols, t->ids,
                     t->koff, t->nl, T, t->kscale);
  hipLaunchKernelGGL(k_tile_red_pack, dim3(chunks, members), dim3(256), 0, st, t->Kw, t->ncol, t->cols, t->ids,
                     t->koff, t->nl, t->woff, t->kscale, t->W16, T);
  CGM_HIP(hipGetLastError());
  CGM_HIP(hipStreamSynchronize(st));  // the host vectors are read by the copies above
  release_factor_workspace(t);  // FP32 matrices: twice the bytes of W, needed only here
  return CGM_SUCCESS;
}

}  // namespace

namespace cgm {

cgm_context* tiles_context(const cgm_tiles* t) { return t->ctx; }
int tiles_maps(const cgm_tiles* t) { return t->maps; }

// Algorithmic bytes of one application to nsys systems: the inverse entries
// streamed (dense form: every entry of every tile in FP32, once per system or
// once per group of eight (T = 8: four) right-hand sides of one map; reduced form: the FP16
// entries of W, once per system or once per group of sixteen right-hand sides
// of one map) plus v in and z out.
double apply_bytes(const cgm_tiles* tl, int nsys) {
  double e = 0.0;
  if (tl->reduced) {
    if (tl->maps == 1)
      e = tl->kept[0] * 4.0 * ((nsys + 15) / 16);
    else
      for (int s = 0; s < nsys; ++s) e += tl->kept[s] * 4.0;
  } else {
    const int group = tl->maps == 1 ? dense_group(tl->M2, nsys) : 1;
    const int streams = (nsys + group - 1) / group;
    if (tl->maps == 1)
      e = tl->kept[0] * 8.0 * streams;
    else
      for (int s = 0; s < nsys; ++s) e += tl->kept[s] * 8.0;
  }
  return e + 16.0 * tl->N * tl->N * nsys;
}

int tiles_apply_io(const cgm_tiles* tl, hipStream_t st, const FnoIO& io, int nsys, const int* done, long sd) {
  if (tl->maps < 1) {
    cgm_set_last_error("the tile preconditioner has not been factored");
    return CGM_ERROR_INVALID_VALUE;
  }
  if (tl->maps > 1 && nsys > tl->maps) {
    cgm_set_last_error("%d systems but %d factored maps", nsys, tl->maps);
    return CGM_ERROR_INVALID_VALUE;
  }
  // live timing inside a long cycle (cgm_longrec_timing): events around the
  // streaming kernel (k_tile_apply, or k_tile_ws of the reduced form) and the
  // application's algorithmic bytes
  LrTiming* tm = tl->ctx->lrt.on ? &tl->ctx->lrt : nullptr;
  const int sl = tm ? tm->cur : -1;
  constexpr int KK = LrTiming::kKernels;
  hipEvent_t* ev = sl >= 0 ? &tm->ev[2 * KK * sl + 4] : nullptr;
  if (ev && !tl->reduced) CGM_HIP(hipEventRecord(ev[0], st));
  int rc;
  switch (tl->M2) {
    case 64: rc = launch_apply_m<64>(tl, st, io, done, sd, nsys); break;
    case 256: rc = launch_apply_m<256>(tl, st, io, done, sd, nsys); break;
    case 1024: rc = launch_apply_m<1024>(tl, st, io, done, sd, nsys); break;
    case 4096:
    case 16384: rc = launch_apply_red(tl, st, io, done, sd, nsys, ev); break;
    default:
      cgm_set_last_error("tile side %d unsupported", tl->T);
      return CGM_ERROR_UNSUPPORTED;
  }
  if (ev && !rc) {
    if (!tl->reduced) CGM_HIP(hipEventRecord(ev[1], st));
    tm->slot_bytes[2][sl] = apply_bytes(tl, nsys);
    tm->slot_has[2][sl] = true;
  }
  return rc;
}

}  // namespace cgm

extern "C" int cgm_tiles_create(cgm_ctx_t c, int T, int batch, cgm_tiles_t* out) {
  CGM_CHECK(c && out, CGM_ERROR_INVALID_VALUE, "null argument");
  *out = nullptr;
  CGM_CHECK(T == 8 || T == 16 || T == 32 || T == 64 || T == 128, CGM_ERROR_UNSUPPORTED,
            "tile side %d: 8, 16, 32, 64 or 128 supported", T);
  CGM_CHECK(c->N % T == 0, CGM_ERROR_UNSUPPORTED, "N=%d is not a multiple of the tile side %d", c->N, T);
  CGM_CHECK(batch >= 1, CGM_ERROR_INVALID_VALUE, "batch %d < 1", batch);
  CGM_HIP(hipSetDevice(c->device));
  cgm_tiles* t = new cgm_tiles();
  t->ctx = c;
  t->device = c->device;
  t->N = c->N;
  t->T = T;
  t->B = batch;
  t->nt = c->N / T;
  t->M2 = T * T;
  t->reduced = T >= 64;
  const size_t ntiles = (size_t)t->nt * t->nt;
  const size_t M2 = (size_t)t->M2;
  bool ok = rocblas_create_handle(&t->h) == rocblas_status_success;
  size_t want = 0;
  auto alloc = [&](void** p, size_t b) {
    if (ok && hipMalloc(p, b) != hipSuccess) ok = false;
    want += b;
  };
  if (!t->reduced) {
    alloc((void**)&t->K, sizeof(float2) * M2 * M2 * ntiles * batch);
    alloc((void**)&t->ipiv, sizeof(int) * M2 * ntiles * batch);
    alloc((void**)&t->info, sizeof(int) * ntiles * batch);
  } else {
    const size_t nb = ntiles * batch;
    alloc((void**)&t->ncol, sizeof(int) * nb);
    alloc((void**)&t->cols, sizeof(unsigned short) * M2 * nb);
    alloc((void**)&t->woff, sizeof(long) * nb);
    alloc((void**)&t->kscale, sizeof(float) * nb);
    alloc((void**)&t->ids, sizeof(int) * nb);
    alloc((void**)&t->koff, sizeof(long) * nb);
    alloc((void**)&t->bloc, sizeof(int) * nb);
    alloc((void**)&t->sloc, sizeof(int) * nb);
    alloc((void**)&t->sstart, sizeof(int) * batch);
    alloc((void**)&t->scount, sizeof(int) * batch);
    alloc((void**)&t->ssize, sizeof(int) * batch);
    alloc((void**)&t->nl, sizeof(int) * nb);
    alloc((void**)&t->info, sizeof(int) * nb);
    if (ok && plan_init(t->P, T) != CGM_SUCCESS) ok = false;
    const size_t M = (size_t)t->P.M;
    alloc((void**)&t->tw32, sizeof(float2) * M);
    alloc((void**)&t->tw64, sizeof(double2) * M);
    alloc((void**)&t->blkT, sizeof(double2) * M2);
    alloc((void**)&t->gq, sizeof(float2) * (M / 2 + 1) * (M / 2 + 1));
    if (ok && upload_twiddles(t) != CGM_SUCCESS) ok = false;
  }
  t->bytes = want;
  if (ok && t->reduced && ensure_scratch(t, batch) != CGM_SUCCESS) ok = false;
  if (!ok) {
    cgm_tiles_destroy(t);
    cgm_set_last_error("cgm_tiles_create: allocation failed (%zu MiB)", want >> 20);
    return CGM_ERROR_ALLOC;
  }
  *out = t;
  return CGM_SUCCESS;
}

extern "C" int cgm_tiles_destroy(cgm_tiles_t t) {
  if (!t) return CGM_SUCCESS;
  (void)hipSetDevice(t->device);
  void* ptrs[] = {t->K,    t->ipiv, t->info, t->ncol, t->cols, t->woff, t->kscale,
                  t->ids,  t->bloc, t->sloc, t->stab, t->spos, t->sstart, t->scount, t->ssize,
                  t->Pw,   t->Xs,   t->xinv, t->koff, t->nl,
                  t->W16,  t->Kw,   t->Pb,    t->Rw,   t->Cw,
                  t->U,    t->Tm,   t->tw32, t->tw64, t->blkT,  t->gq};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (t->h) (void)rocblas_destroy_handle(t->h);
  delete t;
  return CGM_SUCCESS;
}

extern "C" int cgm_tiles_memory(cgm_tiles_t t, size_t* bytes) {
  CGM_CHECK(t && bytes, CGM_ERROR_INVALID_VALUE, "null argument");
  *bytes = t->bytes;
  return CGM_SUCCESS;
}

extern "C" int cgm_tiles_factor(cgm_tiles_t t, const cgm_complex128* block, const float* chi, long chi_stride,
                                int maps) {
  CGM_CHECK(t && block && chi, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(maps >= 1 && maps <= t->B, CGM_ERROR_INVALID_VALUE, "maps %d outside [1, %d]", maps, t->B);
  CGM_CHECK(maps == 1 || chi_stride >= (long)t->N * t->N, CGM_ERROR_INVALID_VALUE,
            "chi_stride must be >= N*N for several maps");
  cgm_context* c = t->ctx;
  CGM_HIP(hipSetDevice(c->device));
  const int ntiles = t->nt * t->nt;
  const int M2 = t->M2;
  t->maps = 0;
  t->kept.assign(maps, 0.0);
  CGM_CHECK(rocblas_set_stream(t->h, c->stream) == rocblas_status_success, CGM_ERROR_DEVICE,
            "rocblas_set_stream failed");
  if (t->reduced) {
    const int rc = factor_reduced(t, (const double2*)block, chi, maps == 1 ? 0 : chi_stride, maps);
    if (rc) return rc;
    CGM_HIP(hipStreamSynchronize(c->stream));
    t->maps = maps;
    return CGM_SUCCESS;
  }
  const int chunks = (int)(((long)M2 * M2 + kBuildChunk - 1) / kBuildChunk);
  hipLaunchKernelGGL(k_tile_build, dim3(ntiles * chunks, maps), dim3(256), 0, c->stream, (const double2*)block, chi,
                     chi_stride, t->K, t->N, t->T, chunks);
  CGM_HIP(hipGetLastError());
  const rocblas_stride sA = (rocblas_stride)M2 * M2;
  const int nb = ntiles * maps;
  rocblas_status s = rocsolver_cgetrf_strided_batched(t->h, M2, M2, (rocblas_float_complex*)t->K, M2, sA, t->ipiv,
                                                      M2, t->info, nb);
  CGM_CHECK(s == rocblas_status_success, CGM_ERROR_DEVICE, "rocsolver getrf: status %d", (int)s);
  std::vector<int> info(nb);
  CGM_HIP(hipMemcpyAsync(info.data(), t->info, sizeof(int) * nb, hipMemcpyDeviceToHost, c->stream));
  CGM_HIP(hipStreamSynchronize(c->stream));
  for (int k = 0; k < nb; ++k)
    CGM_CHECK(info[k] == 0, CGM_ERROR_NONFINITE, "tile %d of map %d is singular (pivot %d)", k % ntiles,
              k / ntiles, info[k]);
  s = rocsolver_cgetri_strided_batched(t->h, M2, (rocblas_float_complex*)t->K, M2, sA, t->ipiv, M2, t->info, nb);
  CGM_CHECK(s == rocblas_status_success, CGM_ERROR_DEVICE, "rocsolver getri: status %d", (int)s);
  CGM_HIP(hipStreamSynchronize(c->stream));
  t->kept.assign(maps, (double)ntiles * M2 * M2);
  t->maps = maps;
  return CGM_SUCCESS;
}

extern "C" int cgm_tiles_apply_bytes(cgm_tiles_t t, int batch, double* bytes) {
  CGM_CHECK(t && bytes, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(t->maps >= 1, CGM_ERROR_INVALID_VALUE, "cgm_tiles_factor has not run");
  CGM_CHECK(batch >= 1 && (t->maps == 1 || batch <= t->maps), CGM_ERROR_INVALID_VALUE,
            "batch %d: %d maps were factored", batch, t->maps);
  *bytes = apply_bytes(t, batch);
  return CGM_SUCCESS;
}

extern "C" int cgm_tiles_apply(cgm_tiles_t t, const cgm_complex64* x, cgm_complex64* y, int batch) {
  CGM_CHECK(t && x && y, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(t->maps >= 1, CGM_ERROR_INVALID_VALUE, "cgm_tiles_factor has not run");
  CGM_CHECK(batch >= 1 && (t->maps == 1 || batch <= t->maps), CGM_ERROR_INVALID_VALUE,
            "batch %d: %d maps were factored", batch, t->maps);
  CGM_CHECK(x != y, CGM_ERROR_INVALID_VALUE, "x and y must not alias");
  CGM_HIP(hipSetDevice(t->device));
  FnoIO io;
  io.v = (const float2*)x;
  io.sV = (long)t->N * t->N;
  io.z = (float2*)y;
  io.sZ = io.sV;
  return tiles_apply_io(t, t->ctx->stream, io, batch, nullptr, 0);
}

// ---------------------------------------------------------------------------
// diagnostics: the application alone on synthetic inverses
// ---------------------------------------------------------------------------
namespace {
// Synthetic dense inverses of one map.
__global__ void k_tile_fill(float2* __restrict__ K, long total) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const float v = 1e-3f * (float)(e % 7);
    K[e] = make_float2(v, -v);
  }
}

// Synthetic reduced form of one map in which every cell carries chi != 0
// (n_t = T^2 for every tile): W16 (total entries), unit scales, identity
// cell lists.
__global__ void k_tile_fill_red(__half2* __restrict__ W16, long total, float* __restrict__ sc, int* __restrict__ ncol,
                                unsigned short* __restrict__ cols, int M2, long ntiles) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const float v = 1e-3f * (float)(e % 7);
    W16[e] = __floats2half2_rn(v, -v);
    if (e < ntiles) {
      sc[e] = 1.f;
      ncol[e] = M2;
    }
    if (e < ntiles * M2) cols[e] = (unsigned short)(e % M2);
  }
}
}  // namespace

extern "C" int cgm_profile_tiles(cgm_tiles_t t, int reps, float* ms) {
  CGM_CHECK(t && ms, CGM_ERROR_INVALID_VALUE, "null argument");
  CGM_CHECK(reps >= 1, CGM_ERROR_INVALID_VALUE, "reps < 1");
  cgm_context* c = t->ctx;
  CGM_HIP(hipSetDevice(c->device));
  const long ntiles = (long)t->nt * t->nt;
  const long total = (long)t->M2 * t->M2 * ntiles;  // one map
  t->maps = 0;
  if (t->reduced) {
    const int rc = layout_reduced(t, std::vector<int>(ntiles, t->M2), 1);
    if (rc) return rc;
    hipLaunchKernelGGL(k_tile_fill_red, dim3(4096), dim3(256), 0, c->stream, t->W16, (long)t->kept[0], t->kscale,
                       t->ncol, t->cols, t->M2, ntiles);
  } else {
    hipLaunchKernelGGL(k_tile_fill, dim3(4096), dim3(256), 0, c->stream, t->K, total);
    t->kept.assign(1, (double)total);
  }
  CGM_HIP(hipGetLastError());
  const long n = (long)t->N * t->N;
  float2 *x = nullptr, *y = nullptr;
  CGM_HIP(hipMalloc((void**)&x, sizeof(float2) * n));
  if (hipMalloc((void**)&y, sizeof(float2) * n) != hipSuccess) {
    (void)hipFree(x);
    cgm_set_last_error("cgm_profile_tiles: allocation failed");
    return CGM_ERROR_ALLOC;
  }
  int rc = CGM_SUCCESS;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (hipMemsetAsync(x, 0, sizeof(float2) * n, c->stream) != hipSuccess || hipEventCreate(&e0) != hipSuccess ||
      hipEventCreate(&e1) != hipSuccess) {
    rc = CGM_ERROR_DEVICE;
  } else {
    t->maps = 1;
    FnoIO io;
    io.v = x;
    io.sV = n;
    io.z = y;
    io.sZ = n;
    rc = tiles_apply_io(t, c->stream, io, 1, nullptr, 0);
    (void)hipEventRecord(e0, c->stream);
    for (int r = 0; !rc && r < reps; ++r) rc = tiles_apply_io(t, c->stream, io, 1, nullptr, 0);
    (void)hipEventRecord(e1, c->stream);
    (void)hipEventSynchronize(e1);
    (void)hipEventElapsedTime(ms, e0, e1);
    *ms /= reps;
    t->maps = 0;  // the synthetic inverses must be factored before use
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(x);
  (void)hipFree(y);
  return rc;
}
