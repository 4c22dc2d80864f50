// Tiled sparse block factorisation A = L D L^T (xg_tileplan.h), the exact
// preconditioner of the PCG under the static integrators.
//
// D holds the inverse of every column's diagonal block as it is eliminated,
// the off-diagonal tiles keep A(i, k) as updated so far beside G(i, k) =
// A(i, k) D_k.  A column's update of tile (i, j) is then one product,
// A(i, j) -= G(i, k) A(j, k)^T, and the sweeps need no triangular solve:
//   forward   y_i -= G(i, k) y_k          (columns up)
//   backward  x_k  = D_k y_k - sum_i G(i, k)^T x_i   (columns down, a level's
//             row tiles i handed on to every column that holds them)
// so a dependent step of a sweep is one 64 x 64 product with a vector.
//
// All products run on the matrix cores (v_mfma_f64_16x16x4: lane l holds
// A[l % 16][l / 16], B[l / 16][l % 16] and rows l / 16 + 4 r, column l % 16 of
// the result) from tiles staged in LDS with rows of 66 doubles, so that
// the 32 lanes of a read phase fall on 32 different 8-byte banks.
//
// The factorisation is bound by its chain of dependent launches, two per
// level, except where a level has hundreds of updates, which the matrix
// cores bound (4,096 cycles a tile).  Against a band factor in 64 x 64 tiles
// with triangular sweeps (one launch per tile column, 41 us each, and two
// more per column and application): 10 x 10 x 20 frame, 14,520 equations,
// 227 tile columns there and 37 levels here, two pushover steps 170 -> 21 ms;
// 150 x 37 quad strip, three steps, 210 -> 13.5 ms; 12^3 bricks 42 -> 7.3 ms;
// a 4 x 3 x 7 frame of force-based elements (840 equations, block Jacobi in
// one workgroup before) 187 -> 4.5 ms.
#include <algorithm>

#include "../../include/xara_gpu.h"
#include "xg_common.h"
#include "xg_kernels.h"
#include "xg_tiles.h"

namespace xg {

namespace {

constexpr int TB = 64;
constexpr int TS = TB * TB;
constexpr int SK = TB + 2;  // LDS row stride of a tile
constexpr int PW = 8;       // columns of a panel
constexpr int SP = 10;      // LDS row stride of a panel
constexpr int HC = 32;      // columns of a half tile
constexpr int SH = HC + 2;  // LDS row stride of a half tile

typedef double d4 __attribute__((ext_vector_type(4)));

// 1/a: the hardware estimate and two Newton steps
__device__ __forceinline__ double rcp_nr(double a) {
  double y = __builtin_amdgcn_rcp(a);
  y = fma(y, fma(-a, y, 1.0), y);
  y = fma(y, fma(-a, y, 1.0), y);
  return y;
}

// orders the compiler only: LDS accesses of one wavefront run in order
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(256) void k_tl_zero(long long total, double2* __restrict__ a) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256)
    a[i] = make_double2(0.0, 0.0);
}

// CSR values into the tiles of the lower block triangle (diagonal tiles
// whole), 8 lanes per row; ones on the padded diagonal of the last panel.
// An entry whose tile the plan does not hold sets bad.
__global__ __launch_bounds__(256) void k_tl_gather(int n, TileView V, const int* __restrict__ rowptr,
                                                   const int* __restrict__ colind, const double* __restrict__ vals,
                                                   double* __restrict__ A, int* __restrict__ bad) {
  const int g = blockIdx.x * 32 + threadIdx.x / 8, lane = threadIdx.x % 8;
  if (g < V.nt && lane == 0) {
    const int w = V.wid[g];
    double* D = A + ((long long)V.colptr[g] + g) * TS;
    for (int i = w; i < (w + 15) / 16 * 16; i++) D[i * TB + i] = 1.0;
  }
  if (g >= n) return;
  const int pr = V.pos[g], tr = pr / TB;
  for (int q = rowptr[g] + lane; q < rowptr[g + 1]; q += 8) {
    const int pc = V.pos[colind[q]], tc = pc / TB;
    if (tc > tr) continue;
    long long slot = (long long)V.colptr[tc] + tc;
    if (tc < tr) {
      int lo = V.colptr[tc], hi = V.colptr[tc + 1];
      const int b = lo, e = hi;
      while (lo < hi) {
        const int m = (lo + hi) / 2;
        if (V.row[m] < tr) lo = m + 1;
        else hi = m;
      }
      if (lo >= e || V.row[lo] != tr) {
        atomicExch(bad, 2);
        continue;
      }
      slot += 1 + lo - b;
    }
    A[slot * TS + (pr % TB) * TB + pc % TB] = vals[q];
  }
}

// tile (row-major, 64 wide) columns 0 .. kc-1 to registers and to LDS; 256
// threads, thread t columns 2 (t % 32) .. of rows t / 32 + 8 i
__device__ __forceinline__ void tile_get(double2 (&v)[8], const double* __restrict__ g, int kc) {
  const int c = 2 * (threadIdx.x % 32), r = threadIdx.x / 32;
#pragma unroll
  for (int i = 0; i < 8; i++)
    v[i] = c < kc ? *reinterpret_cast<const double2*>(g + (r + 8 * i) * TB + c) : make_double2(0.0, 0.0);
}
__device__ __forceinline__ void tile_put(double* s, const double2 (&v)[8]) {
  const int c = 2 * (threadIdx.x % 32), r = threadIdx.x / 32;
#pragma unroll
  for (int i = 0; i < 8; i++) *reinterpret_cast<double2*>(s + (r + 8 * i) * SK + c) = v[i];
}

// acc += sign * X Y^T over kc columns: wavefront w the 32 x 32 quadrant (w / 2,
// w % 2) as 2 x 2 blocks, X and Y in LDS (rows of S doubles)
template <bool NEG, int S>
__device__ __forceinline__ void quad_gemm(d4 (&acc)[2][2], const double* X, const double* Y, int kc) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const double* x0 = X + (32 * (w >> 1) + (l & 15)) * S + (l >> 4);
  const double* y0 = Y + (32 * (w & 1) + (l & 15)) * S + (l >> 4);
  for (int k = 0; k < kc; k += 16) {
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const double a0 = NEG ? -x0[k + i] : x0[k + i], a1 = NEG ? -x0[16 * S + k + i] : x0[16 * S + k + i];
      const double b0 = y0[k + i], b1 = y0[16 * S + k + i];
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
  }
}
__device__ __forceinline__ void quad_load(d4 (&acc)[2][2], const double* __restrict__ g) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        acc[a][b][r] = g[(32 * (w >> 1) + 16 * a + (l >> 4) + 4 * r) * TB + 32 * (w & 1) + 16 * b + (l & 15)];
}
__device__ __forceinline__ void quad_store(double* __restrict__ g, const d4 (&acc)[2][2]) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        g[(32 * (w >> 1) + 16 * a + (l >> 4) + 4 * r) * TB + 32 * (w & 1) + 16 * b + (l & 15)] = acc[a][b][r];
}

// The value of lane C of the lane's row of 16
template <int C>
__device__ __forceinline__ double row_d(double v) {
  const long long b = __double_as_longlong(v);
  return __longlong_as_double(__builtin_amdgcn_update_dpp(b, b, 0x150 + C, 0xf, 0xf, true));
}

// One pivot (row g0 + C, in lane C of every 16, its column at a[C]) of the
// symmetric sweep over a panel of PW columns, the lane holding row `row` of
// the panel: every other row takes its multiple of the pivot row off, the
// pivot row is left unscaled (its lane multiplies it by 1/pivot after the
// panel, which commutes with the later row operations).
template <int C>
__device__ __forceinline__ void sweep_pivot(double (&a)[PW], double& scale, int row, int g0) {
  const double inv = rcp_nr(row_d<C>(a[C]));
  const bool own = row == g0 + C;
  const double u = own ? 0.0 : a[C] * inv;
  if (own) scale = inv;
#pragma unroll
  for (int j = 0; j < PW; j++)
    if (j != C) a[j] = fma(-u, row_d<C>(a[j]), a[j]);
  // (u is 0 in the pivot's own lane: one half of -1)
  a[C] = __hiloint2double(own ? 0xbff00000 : __double2hiint(u), __double2loint(u));
}

// What a panel leaves to be done after the next barrier: the products of
// blocks 1 .. 3 (as numbered then), A operand a, B operands b
struct Pending {
  double a[2], b[3][2];
};

// One panel, columns 16 p + 8 H .., of the symmetric sweep: m[J] the block
// (w, (p + J) % 4) of the wavefront's block row.  P holds the panel's
// columns, Wp the last panel as swept, W takes this one, Pn the next panel.
template <int H>
__device__ __forceinline__ void panel_step(d4 (&m)[4], double* P, double* Pn, double* W, const double* Wp, int p,
                                           int w, bool& nonpos, Pending& q) {
  constexpr int HP = 1 - H, E = H;  // E: the block that holds the next panel
  const int l = threadIdx.x & 63, lc = l & 15, lr = l >> 4;
  const int g0 = 16 * p + 8 * H, row = lc < 8 ? g0 + lc : 16 * w + 8 * (lr & 1) + lc - 8;
  __syncthreads();
  double a[PW], v[4][2], vm[4], b[4][2];
#pragma unroll
  for (int j = 0; j < PW; j += 2) {
    const double2 x = *reinterpret_cast<const double2*>(P + row * SP + j);
    a[j] = x.x;
    a[j + 1] = x.y;
  }
#pragma unroll
  for (int J = 0; J < 4; J++) {
    const int c = (16 * ((p + J) & 3) + lc) * SP + lr;
    v[J][0] = Wp[c];
    v[J][1] = Wp[c + 4];
    b[J][0] = P[c];
    b[J][1] = P[c + 4];
  }
  if (H == 0)
#pragma unroll
    for (int r = 0; r < 4; r++) vm[r] = Wp[(16 * w + lr + 4 * r) * SP + (lc & 7)];
  // the last panel's products, while this one comes from LDS
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int J = 1; J < 4; J++) m[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.a[k], q.b[J - 1][k], m[J], 0, 0, 0);
  double scale = 1.0;
  sweep_pivot<0>(a, scale, row, g0);
  sweep_pivot<1>(a, scale, row, g0);
  sweep_pivot<2>(a, scale, row, g0);
  sweep_pivot<3>(a, scale, row, g0);
  sweep_pivot<4>(a, scale, row, g0);
  sweep_pivot<5>(a, scale, row, g0);
  sweep_pivot<6>(a, scale, row, g0);
  sweep_pivot<7>(a, scale, row, g0);
  // the last panel's columns and rows (registers 2 HP and 2 HP + 1 of its
  // block row) from the panel as swept; the next panel's block had its
  // columns, and for H = 1 its rows, before
  if (H == 0) {
    const bool swept = p > 0 && (lc >> 3) == HP;
#pragma unroll
    for (int r = 0; r < 4; r++) m[3][r] = swept ? vm[r] : m[3][r];
  }
  const bool prow = w == (H == 0 ? p - 1 : p);
#pragma unroll
  for (int J = H == 0 ? 0 : 1; J < 4; J++) {
    m[J][2 * HP] = prow ? v[J][0] : m[J][2 * HP];
    m[J][2 * HP + 1] = prow ? v[J][1] : m[J][2 * HP + 1];
  }
  // a pivot that is not positive (or not a number): the caller drops the
  // whole factor, so what follows from it does not matter
  nonpos |= !(scale > 0.0) || !isfinite(scale);
  if (lc >= 8 && lr < 2)
#pragma unroll
    for (int j = 0; j < PW; j += 2)
      *reinterpret_cast<double2*>(W + row * SP + j) = make_double2(a[j] * scale, a[j + 1] * scale);
  wave_order();
  // block (I, J) -= W_I P_J^T: the next panel's now
  q.a[0] = -W[(16 * w + lc) * SP + lr];
  q.a[1] = -W[(16 * w + lc) * SP + 4 + lr];
  m[E] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.a[0], b[E][0], m[E], 0, 0, 0);
  m[E] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.a[1], b[E][1], m[E], 0, 0, 0);
#pragma unroll
  for (int J = 1; J < 4; J++)
#pragma unroll
    for (int k = 0; k < 2; k++) q.b[J - 1][k] = b[(J + E) & 3][k];
  if (H == 0) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const double x = W[(16 * w + lr + 4 * r) * SP + (lc & 7)];
      m[0][r] = lc < 8 ? x : m[0][r];
    }
    m[0][0] = w == p ? -q.a[0] : m[0][0];
    m[0][1] = w == p ? -q.a[1] : m[0][1];
    if (lc >= 8)
#pragma unroll
      for (int r = 0; r < 4; r++) Pn[(16 * w + lr + 4 * r) * SP + lc - 8] = m[0][r];
  } else {
    // this panel's rows of the next, from the wavefront that swept them as
    // its columns
    if (lc < 8)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (r < 2 || w != p) Pn[(16 * w + lr + 4 * r) * SP + lc] = m[1][r];
    if (w == ((p + 1) & 3)) Pn[(16 * p + 8 + (l >> 3)) * SP + (l & 7)] = W[(16 * w + (l & 7)) * SP + (l >> 3)];
  }
}

// Task {column k, first row tile, row tiles} of a level: the inverse of the
// diagonal block, in every workgroup of the column, by the symmetric sweep
// in panels of 8 columns (wavefront w keeps block row w of 16 x 16 blocks in
// accumulators and sweeps its 16 rows of the panel, the 8 pivot rows beside
// them in every 16 lanes, so one barrier per panel), then G(i, k) = A(i, k)
// D_k for its row tiles.  The first workgroup of a column stores D_k.
//
// Bound by the pivots' chain and the passage of a panel through LDS.  A
// pivot row reaches the other lanes by one DPP move a value, and of the
// products after a panel only the next panel's block is waited for; the
// others fill the wait for its columns.  Of the 24,100 cycles of the sweep
// 141 go to each of 64 pivots.  Panels of 8 balance the pivots against the
// products.  One column with one row tile, launch to launch: 15.7 us (19.2
// when every wavefront swept all 64 rows, pivot rows by readlane, 224 cycles
// a pivot, with all products before the next panel; 16.1 with the products
// held between the pivots; the 4 x 4 register-blocked band factor before
// took 41 per tile column).
__global__ __launch_bounds__(256) void k_tl_panel(TileView V, const int4* __restrict__ task,
                                                  const double* __restrict__ A, double* __restrict__ G,
                                                  int* __restrict__ bad) {
  __shared__ __align__(16) double sh[2 * TB * SK];
  double *P0 = sh, *P1 = sh + TB * SP, *W0 = sh + 2 * TB * SP, *W1 = sh + 3 * TB * SP;
  const int4 t = task[blockIdx.x];
  // the wavefront's number as a scalar: matrix instructions ignore the lane
  // mask, so the branch on it has to be a jump
  const int k = t.x, l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long dslot = (long long)V.colptr[k] + k;
  const int np = (V.wid[k] + 15) / 16;
  d4 m[4];
  {
    const double* D = A + dslot * TS;
#pragma unroll
    for (int J = 0; J < 4; J++)
#pragma unroll
      for (int r = 0; r < 4; r++) m[J][r] = D[(16 * w + (l >> 4) + 4 * r) * TB + 16 * J + (l & 15)];
  }
  double2 x[8];
  if (t.z > 0) tile_get(x, A + (dslot + 1 + t.y) * TS, 16 * np);
  bool nonpos = false;
  const int lc = l & 15, lr = l >> 4;
  if (lc < 8)
#pragma unroll
    for (int r = 0; r < 4; r++) P0[(16 * w + lr + 4 * r) * SP + lc] = m[0][r];
  Pending q = {};
  // the block column in work is m[0]: after each one the blocks move round
  // by one, and everything in the loop is straight-line code (branches on
  // the block column made the compiler copy all accumulators at every one:
  // 42 us)
#pragma unroll 1
  for (int p = 0; p < np; p++) {
    panel_step<0>(m, P0, P1, W0, W1, p, w, nonpos, q);
    panel_step<1>(m, P1, P0, W1, W0, p, w, nonpos, q);
    const d4 m0 = m[0];
    m[0] = m[1];
    m[1] = m[2];
    m[2] = m[3];
    m[3] = m0;
  }
  // what the last panel left
  __syncthreads();
#pragma unroll
  for (int J = 0; J < 4; J++) {
    if (J > 0) {
      m[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.a[0], q.b[J > 0 ? J - 1 : 0][0], m[J], 0, 0, 0);
      m[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.a[1], q.b[J > 0 ? J - 1 : 0][1], m[J], 0, 0, 0);
    }
    const int c = (16 * ((np + J) & 3) + lc) * SP + lr;
    if (J == 3)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const double v = W1[(16 * w + lr + 4 * r) * SP + (lc & 7)];
        m[3][r] = lc >= 8 ? v : m[3][r];
      }
    const double v0 = W1[c], v1 = W1[c + 4];
    m[J][2] = w == np - 1 ? v0 : m[J][2];
    m[J][3] = w == np - 1 ? v1 : m[J][3];
  }
  if (nonpos && t.y == 0 && w == 0) atomicExch(bad, 1);
  __syncthreads();
  // D = -m, zero outside the column's panels
  double* X = sh;
  double* D = sh + TB * SK;
#pragma unroll
  for (int J = 0; J < 4; J++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int Jc = (np + J) & 3, i = 16 * w + lr + 4 * r, c = 16 * Jc + lc;
      const double v = (w < np && Jc < np) ? -m[J][r] : 0.0;
      D[i * SK + c] = v;
      if (t.y == 0) G[dslot * TS + i * TB + c] = v;
    }
  for (int j = 0; j < t.z; j++) {
    const long long slot = dslot + 1 + t.y + j;
    tile_put(X, x);
    __syncthreads();
    if (j + 1 < t.z) tile_get(x, A + (slot + 1) * TS, 16 * np);
    d4 acc[2][2] = {};
    quad_gemm<false, SK>(acc, X, D, 16 * np);  // D is symmetric
    quad_store(G + slot * TS, acc);
    __syncthreads();
  }
}

// half tile (columns 32 h ..) of a row-major tile to registers and LDS, 256
// threads, thread t columns 2 (t % 16) .. of rows t / 16 + 16 i
__device__ __forceinline__ void half_get(double2 (&v)[4], const double* __restrict__ g, int kc) {
  const int c = 2 * (threadIdx.x % 16), r = threadIdx.x / 16;
#pragma unroll
  for (int i = 0; i < 4; i++)
    v[i] = c < kc ? *reinterpret_cast<const double2*>(g + (r + 16 * i) * TB + c) : make_double2(0.0, 0.0);
}
__device__ __forceinline__ void half_put(double* s, const double2 (&v)[4]) {
  const int c = 2 * (threadIdx.x % 16), r = threadIdx.x / 16;
#pragma unroll
  for (int i = 0; i < 4; i++) *reinterpret_cast<double2*>(s + (r + 16 * i) * SH + c) = v[i];
}

// One target tile of a level's updates: A(target) -= sum of G(i, k) A(j, k)^T
// over the level's columns k that reach it, in ascending order.  Half tiles
// are staged, so that four workgroups fit a compute unit and one's loads
// run under another's products (whole tiles, two workgroups a unit:
// slower, figures at tiles_factor).
__global__ __launch_bounds__(256) void k_tl_update(const int* __restrict__ tgt, const int* __restrict__ src,
                                                   const int* __restrict__ sg, const int* __restrict__ sa,
                                                   const int* __restrict__ sk, double* __restrict__ A,
                                                   const double* __restrict__ G) {
  __shared__ __align__(16) double X[TB * SH];
  __shared__ __align__(16) double Y[TB * SH];
  const int b = src[blockIdx.x], e = src[blockIdx.x + 1];
  double* T = A + (long long)tgt[blockIdx.x] * TS;
  double2 x[4], y[4];
  int s = b, c0 = 0, kc = sk[b];
  half_get(x, G + (long long)sg[b] * TS, kc);
  half_get(y, A + (long long)sa[b] * TS, kc);
  d4 acc[2][2];
  quad_load(acc, T);
  while (true) {
    half_put(X, x);
    half_put(Y, y);
    __syncthreads();
    const int now = kc - c0 < HC ? kc - c0 : HC;
    if (c0 + HC < kc) {
      c0 += HC;
    } else {
      s++;
      c0 = 0;
      if (s < e) kc = sk[s];
    }
    if (s < e) {
      half_get(x, G + (long long)sg[s] * TS + c0, kc - c0);
      half_get(y, A + (long long)sa[s] * TS + c0, kc - c0);
    }
    quad_gemm<true, SH>(acc, X, Y, now);
    if (s >= e) break;
    __syncthreads();
  }
  quad_store(T, acc);
}

// The same for a quarter of the target, four workgroups to a tile, whole
// sources staged: for levels with too few targets to fill the chip, where
// the products of one tile follow each other in one compute unit.
__device__ __forceinline__ void quarter_get(double2 (&v)[4], const double* __restrict__ g, int kc) {
  const int c = 2 * (threadIdx.x % 32), r = threadIdx.x / 32;
#pragma unroll
  for (int i = 0; i < 4; i++)
    v[i] = c < kc ? *reinterpret_cast<const double2*>(g + (r + 8 * i) * TB + c) : make_double2(0.0, 0.0);
}
__device__ __forceinline__ void quarter_put(double* s, const double2 (&v)[4]) {
  const int c = 2 * (threadIdx.x % 32), r = threadIdx.x / 32;
#pragma unroll
  for (int i = 0; i < 4; i++) *reinterpret_cast<double2*>(s + (r + 8 * i) * SK + c) = v[i];
}
__global__ __launch_bounds__(256) void k_tl_update_quarter(const int* __restrict__ tgt, const int* __restrict__ src,
                                                           const int* __restrict__ sg, const int* __restrict__ sa,
                                                           const int* __restrict__ sk, double* __restrict__ A,
                                                           const double* __restrict__ G) {
  __shared__ __align__(16) double X[TB / 2 * SK];
  __shared__ __align__(16) double Y[TB / 2 * SK];
  const int t = blockIdx.x >> 2, row = 32 * (blockIdx.x >> 1 & 1), col = 32 * (blockIdx.x & 1);
  const int b = src[t], e = src[t + 1], l = threadIdx.x & 63, w = threadIdx.x >> 6;
  double* T = A + (long long)tgt[t] * TS + (row + 16 * (w >> 1) + (l >> 4)) * TB + col + 16 * (w & 1) + (l & 15);
  const double* x0 = X + (16 * (w >> 1) + (l & 15)) * SK + (l >> 4);
  const double* y0 = Y + (16 * (w & 1) + (l & 15)) * SK + (l >> 4);
  double2 x[4], y[4];
  int kc = sk[b];
  quarter_get(x, G + (long long)sg[b] * TS + row * TB, kc);
  quarter_get(y, A + (long long)sa[b] * TS + col * TB, kc);
  d4 acc;
#pragma unroll
  for (int r = 0; r < 4; r++) acc[r] = T[4 * r * TB];
  for (int s = b; s < e; s++) {
    quarter_put(X, x);
    quarter_put(Y, y);
    __syncthreads();
    const int now = kc;
    if (s + 1 < e) {
      kc = sk[s + 1];
      quarter_get(x, G + (long long)sg[s + 1] * TS + row * TB, kc);
      quarter_get(y, A + (long long)sa[s + 1] * TS + col * TB, kc);
    }
    for (int k = 0; k < now; k += 16)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-x0[k + i], y0[k + i], acc, 0, 0, 0);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 4; r++) T[4 * r * TB] = acc[r];
}

// Sweeps: 1,024 threads per row tile (forward) or column (backward).
// Forward: four sources at a time, 256 threads each (row t / 4, columns
// 16 (t % 4) ..), the partial sums added in order.
template <int R>
__global__ __launch_bounds__(1024) void k_tl_fwd(const int* __restrict__ row, const int* __restrict__ src,
                                                 const int* __restrict__ sg, const int* __restrict__ sc, int npad,
                                                 const double* __restrict__ G, double* __restrict__ Y) {
  __shared__ double part[R][4][TB];
  const int b = src[blockIdx.x], e = src[blockIdx.x + 1];
  const int grp = threadIdx.x >> 8, t = threadIdx.x & 255, r = t >> 2, q = t & 3;
  double acc[R];
#pragma unroll
  for (int i = 0; i < R; i++) acc[i] = 0.0;
  for (int s = b + grp; s < e; s += 4) {
    const double2* g = reinterpret_cast<const double2*>(G + (long long)sg[s] * TS + r * TB);
    const double2* y = reinterpret_cast<const double2*>(Y + (long long)sc[s] * TB);
    double2 gv[8];
    // the quad's lanes read neighbouring 16-byte pieces of the row
#pragma unroll
    for (int j = 0; j < 8; j++) gv[j] = g[4 * j + q];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const double2 v = y[(long long)i * (npad / 2) + 4 * j + q];
        acc[i] = fma(gv[j].x, v.x, acc[i]);
        acc[i] = fma(gv[j].y, v.y, acc[i]);
      }
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    acc[i] += __shfl_xor(acc[i], 1, 64);
    acc[i] += __shfl_xor(acc[i], 2, 64);
    if (q == 0) part[i][grp][r] = acc[i];
  }
  __syncthreads();
  if (threadIdx.x < R * TB) {
    const int i = threadIdx.x / TB, rr = threadIdx.x % TB;
    double* y = Y + (long long)i * npad + (long long)row[blockIdx.x] * TB + rr;
    *y -= ((part[i][0][rr] + part[i][1][rr]) + part[i][2][rr]) + part[i][3][rr];
  }
}

// z_k = D_k y_k for every column
template <int R>
__global__ __launch_bounds__(256) void k_tl_diag(TileView V, int npad, const double* __restrict__ G,
                                                 const double* __restrict__ Y, double* __restrict__ X) {
  const int k = blockIdx.x, r = threadIdx.x >> 2, q = threadIdx.x & 3;
  const double2* g = reinterpret_cast<const double2*>(G + ((long long)V.colptr[k] + k) * TS + r * TB);
  const double2* y = reinterpret_cast<const double2*>(Y + (long long)k * TB);
  double acc[R];
#pragma unroll
  for (int i = 0; i < R; i++) acc[i] = 0.0;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const double2 d = g[4 * j + q];
#pragma unroll
    for (int i = 0; i < R; i++) {
      const double2 v = y[(long long)i * (npad / 2) + 4 * j + q];
      acc[i] = fma(d.x, v.x, acc[i]);
      acc[i] = fma(d.y, v.y, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    acc[i] += __shfl_xor(acc[i], 1, 64);
    acc[i] += __shfl_xor(acc[i], 2, 64);
    if (q == 0) X[(long long)i * npad + (long long)k * TB + r] = acc[i];
  }
}

// Backward: x_k -= sum of G(i, k)^T x_i over the level's row tiles i of column
// k.  Wavefront g takes rows 16 (g % 4) .. of sources g / 4, g / 4 + 4, ...,
// lane c column c.  (The columns of a level pulling all their row tiles at
// once, up to 25 tiles through one compute unit, took 15.8 us a launch on
// the 10 x 10 x 20 frame.)
template <int R>
__global__ __launch_bounds__(1024) void k_tl_bwd(const int* __restrict__ col, const int* __restrict__ src,
                                                 const int* __restrict__ sg, const int* __restrict__ sr, int npad,
                                                 const double* __restrict__ G, double* __restrict__ X) {
  __shared__ double part[R][16][TB];
  const int b = src[blockIdx.x], e = src[blockIdx.x + 1];
  const int g = threadIdx.x >> 6, c = threadIdx.x & 63, r0 = 16 * (g & 3);
  double acc[R];
#pragma unroll
  for (int i = 0; i < R; i++) acc[i] = 0.0;
  for (int s = b + (g >> 2); s < e; s += 4) {
    const double* T = G + (long long)sg[s] * TS + r0 * TB + c;
    const double* v = X + (long long)sr[s] * TB + r0;
    double tv[16];
#pragma unroll
    for (int r = 0; r < 16; r++) tv[r] = T[r * TB];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i] = fma(tv[r], v[(long long)i * npad + r], acc[i]);
  }
#pragma unroll
  for (int i = 0; i < R; i++) part[i][g][c] = acc[i];
  __syncthreads();
  if (threadIdx.x < R * TB) {
    const int i = threadIdx.x / TB, cc = threadIdx.x % TB;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 16; q++) s += part[i][q][cc];
    X[(long long)i * npad + (long long)col[blockIdx.x] * TB + cc] -= s;
  }
}

// y(p) = v(equation at position p), 0 on the padding; and back
__global__ __launch_bounds__(256) void k_tl_in(int npad, const int* __restrict__ ipos, const double* __restrict__ v,
                                               double* __restrict__ y) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= npad) return;
  const int e = ipos[p];
  y[p] = e >= 0 ? v[e] : 0.0;
}
__global__ __launch_bounds__(256) void k_tl_out(int n, const int* __restrict__ pos, const double* __restrict__ x,
                                                double* __restrict__ v) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e < n) v[e] = x[pos[e]];
}

// ---- PCG vectors, one workgroup per right-hand side ----
__device__ __forceinline__ double wg_sum(double v, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0.0;
#pragma unroll
  for (int w = 0; w < 16; w++) r += sh[w];
  return r;
}

// r = b (x = 0), or r = b - q with q = A x from the guess in x (warm)
__global__ __launch_bounds__(1024) void k_tl_start(int n, TilePcg P, double tol2) {
  __shared__ double sh[16];
  const TileRhs& v = P.v[blockIdx.x];
  TileScal& S = P.S[blockIdx.x];
  double bb = 0.0, rr = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const double b = v.b[i], r = v.warm ? b - v.q[i] : b;
    v.r[i] = r;
    bb = fma(b, b, bb);
    rr = fma(r, r, rr);
  }
  bb = wg_sum(bb, sh);
  rr = wg_sum(rr, sh);
  const bool zero = !(bb > 0.0);
  if (!v.warm || zero)
    for (int i = threadIdx.x; i < n; i += 1024) v.x[i] = 0.0;
  if (threadIdx.x == 0) {
    S.bb = bb;
    S.rr = zero ? 0.0 : rr;
    S.rz = 0.0;
    S.iters = 0;
    S.fail = 0;
    S.conv = zero || (v.warm && rr <= tol2 * bb) ? 1 : 0;
  }
}
// r.z, beta, p = z + beta p
__global__ __launch_bounds__(1024) void k_tl_dir(int n, TilePcg P) {
  __shared__ double sh[16];
  const TileRhs& v = P.v[blockIdx.x];
  TileScal& S = P.S[blockIdx.x];
  if (S.conv) return;
  const bool first = S.iters == 0;
  const double old = S.rz;
  double rz = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) rz = fma(v.r[i], v.z[i], rz);
  rz = wg_sum(rz, sh);
  const double beta = first ? 0.0 : rz / old;
  for (int i = threadIdx.x; i < n; i += 1024) v.p[i] = first ? v.z[i] : fma(beta, v.p[i], v.z[i]);
  if (threadIdx.x == 0) S.rz = rz;
}
// p.q, alpha, x += alpha p, r -= alpha q, r.r and the stop test
__global__ __launch_bounds__(1024) void k_tl_step(int n, TilePcg P, double tol2) {
  __shared__ double sh[16];
  const TileRhs& v = P.v[blockIdx.x];
  TileScal& S = P.S[blockIdx.x];
  if (S.conv) return;
  const double rz = S.rz, bb = S.bb;
  double pq = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) pq = fma(v.p[i], v.q[i], pq);
  pq = wg_sum(pq, sh);
  if (pq == 0.0 || !isfinite(pq)) {
    if (threadIdx.x == 0) {
      S.iters++;
      S.conv = S.fail = 1;
    }
    return;
  }
  const double alpha = rz / pq;
  double rr = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) {
    v.x[i] = fma(alpha, v.p[i], v.x[i]);
    const double r = fma(-alpha, v.q[i], v.r[i]);
    v.r[i] = r;
    rr = fma(r, r, rr);
  }
  rr = wg_sum(rr, sh);
  if (threadIdx.x == 0) {
    S.iters++;
    S.rr = rr;
    if (rr <= tol2 * bb) S.conv = 1;
  }
}

}  // namespace

// Levels of up to this many targets are updated in quarter tiles.  Above it
// the chip is full and whole tiles read half as much: 33^3 bricks, levels of
// up to thousands, 137 ms a pass with the line at 512 or 1,024, 145 with
// quarters throughout.  Below it quarters win: 10 x 10 x 20 frame 21.0 ms
// without them, 20.1 with the line at 256, 19.4 at 1,024; 12^3 bricks 6.5,
// 5.9, 5.7; 64 x 16 quad mesh 7.1, 6.4 (a tile of four sources 10.6 -> 8 us).
constexpr int kTileSplit = 1024;
void tiles_factor(hipStream_t s, int n, const TileView& V, const TileHost& H, const int* rowptr, const int* colind,
                  const double* vals, double* A, double* G, int* bad) {
  if (n <= 0) return;
  const long long total = H.tiles * (TS / 2);
  hipLaunchKernelGGL(k_tl_zero, dim3((unsigned)std::min<long long>((total + 255) / 256, 8192)), dim3(256), 0, s, total,
                     reinterpret_cast<double2*>(A));
  hipLaunchKernelGGL(k_tl_gather, dim3((std::max(n, V.nt) + 31) / 32), dim3(256), 0, s, n, V, rowptr, colind, vals, A,
                     bad);
  for (size_t l = 0; l + 1 < H.panptr.size(); l++) {
    hipLaunchKernelGGL(k_tl_panel, dim3(H.panptr[l + 1] - H.panptr[l]), dim3(256), 0, s, V, V.task + H.panptr[l], A, G,
                       bad);
    const int nu = H.upptr[l + 1] - H.upptr[l];
    if (nu > kTileSplit)
      hipLaunchKernelGGL(k_tl_update, dim3(nu), dim3(256), 0, s, V.uptgt + H.upptr[l], V.upsrc + H.upptr[l], V.srcg,
                         V.srca, V.srck, A, G);
    else if (nu > 0)
      hipLaunchKernelGGL(k_tl_update_quarter, dim3(4 * nu), dim3(256), 0, s, V.uptgt + H.upptr[l],
                         V.upsrc + H.upptr[l], V.srcg, V.srca, V.srck, A, G);
  }
}

template <int R>
static void sweeps(hipStream_t s, const TileView& V, const TileHost& H, const double* G, double* Y, double* X) {
  const int npad = V.nt * TB;
  for (size_t l = 0; l + 1 < H.fwptr.size(); l++) {
    const int nf = H.fwptr[l + 1] - H.fwptr[l];
    if (nf > 0)
      hipLaunchKernelGGL(k_tl_fwd<R>, dim3(nf), dim3(1024), 0, s, V.fwrow + H.fwptr[l], V.fwsrc + H.fwptr[l], V.fwg,
                         V.fwk, npad, G, Y);
  }
  hipLaunchKernelGGL(k_tl_diag<R>, dim3(V.nt), dim3(256), 0, s, V, npad, G, Y, X);
  for (int l = (int)H.bwptr.size() - 2; l >= 0; l--) {
    const int nb = H.bwptr[l + 1] - H.bwptr[l];
    if (nb > 0)
      hipLaunchKernelGGL(k_tl_bwd<R>, dim3(nb), dim3(1024), 0, s, V.bwcol + H.bwptr[l], V.bwsrc + H.bwptr[l], V.bwg,
                         V.bwr, npad, G, X);
  }
}

void tiles_sweeps(hipStream_t s, const TileView& V, const TileHost& H, int nrhs, const double* G, double* Y, double* X) {
  if (nrhs == 1) sweeps<1>(s, V, H, G, Y, X);
  else if (nrhs == 2) sweeps<2>(s, V, H, G, Y, X);
  else throw Error(XG_ERR_ARG, "tile sweeps: one or two right-hand sides");
}

void tiles_in(hipStream_t s, const TileView& V, const double* v, double* y) {
  const int npad = V.nt * TB;
  hipLaunchKernelGGL(k_tl_in, dim3((npad + 255) / 256), dim3(256), 0, s, npad, V.ipos, v, y);
}
void tiles_out(hipStream_t s, int n, const TileView& V, const double* x, double* v) {
  hipLaunchKernelGGL(k_tl_out, dim3((n + 255) / 256), dim3(256), 0, s, n, V.pos, x, v);
}
void tiles_pcg_start(hipStream_t s, int n, int nrhs, const TilePcg& P, double tol2) {
  hipLaunchKernelGGL(k_tl_start, dim3(nrhs), dim3(1024), 0, s, n, P, tol2);
}
void tiles_pcg_dir(hipStream_t s, int n, int nrhs, const TilePcg& P) {
  hipLaunchKernelGGL(k_tl_dir, dim3(nrhs), dim3(1024), 0, s, n, P);
}
void tiles_pcg_step(hipStream_t s, int n, int nrhs, const TilePcg& P, double tol2) {
  hipLaunchKernelGGL(k_tl_step, dim3(nrhs), dim3(1024), 0, s, n, P, tol2);
}

}  // namespace xg
