// DispBeamColumn2d/3d over FiberSection2d/3d on gfx950: per-operation
// kernels over a frame group (bodies in xg_frame_impl.h).
#include "xg_frame_impl.h"
#include "xg_kernels.h"

namespace xg {

template <bool D3>
__global__ __launch_bounds__(256) void k_frame_update(FrameDev f, const double* __restrict__ U) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long sec = (long long)blockIdx.x * 4 + wave;
  if (sec >= f.nsec) return;
  section_update<D3>(f, sec, lane, U);
}

// 64 / RW sections of one definition per wavefront (section_rows): rows of
// 16 lanes (four sections, totals by butterfly) or 20 (three sections,
// totals through LDS; held to three waves per SIMD)
template <bool D3>
__global__ __launch_bounds__(256) void k_frame_update_rows(FrameDev f, const double* __restrict__ U) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long w = (long long)blockIdx.x * 4 + wave;
  if (w >= f.nrw) return;
  section_rows<D3, 16>(f, w, lane, U, nullptr);
}
template <bool D3>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_frame_update_rows20(
    FrameDev f, const double* __restrict__ U) {
  constexpr int NV = D3 ? 9 : 5;
  __shared__ double red[4 * NV * 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long w = (long long)blockIdx.x * 4 + wave;
  if (w >= f.nrw) return;
  section_rows<D3, 20>(f, w, lane, U, red + wave * NV * 64);
}

template <bool D3>
__global__ __launch_bounds__(256) void k_frame_revert(FrameDev f) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long sec = (long long)blockIdx.x * 4 + wave;
  if (sec >= f.nsec) return;
  section_revert<D3>(f, sec, lane);
}

// Committed and trial histories of revertToStart (Steel02.cpp:69-95,
// Concrete02.cpp:321-337), one wavefront per section.  Writes only: 387 MB
// on the 10 x 10 x 20 frame.  (Kept on the host and copied from there they
// took 14.7 of the 38.0 ms of that frame's two-step pushover from the start.)
__global__ __launch_bounds__(256) void k_frame_start(FrameDev f) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long sec = (long long)blockIdx.x * 4 + wave;
  if (sec >= f.nsec) return;
  const int def = f.secdef[sec / f.nip];
  for (int fi = f.def_off[def] + lane; fi < f.def_off[def + 1]; fi += 64) {
    const int kind = f.fkind[fi];
    if (kind == 1) {
      const Steel02Param p = f.steelp[f.fmat[fi]];
      const long long n = f.nsteel, k = f.steel_base[sec] + f.flocal[fi];
      const double epsy = p.Fy / p.E0, eps = p.sigini != 0.0 ? p.sigini / p.E0 : 0.0;
      const double h[kSteelHist] = {-epsy, epsy, 0, 0, 0, 0, 0, eps, p.sigini != 0.0 ? p.sigini : 0.0, p.E0};
#pragma unroll
      for (int c = 0; c < kSteelHist; c++) f.st_c[c * n + k] = f.st_t[c * n + k] = h[c];
      f.kon_c[k] = f.kon_t[k] = 0;
    } else if (kind == 2) {
      const Concrete02Param p = f.concp[f.fmat[fi]];
      const long long n = f.nconc, k = f.conc_base[sec] + f.flocal[fi];
      const double h[kConcHist] = {0, 0, 0, 0, 2.0 * p.fc / p.epsc0};
#pragma unroll
      for (int c = 0; c < kConcHist; c++) f.cs_c[c * n + k] = f.cs_t[c * n + k] = h[c];
    } else {
      const long long k = f.elas_base[sec] + f.flocal[fi];
      f.el_c[k] = f.el_t[k] = 0.0;
    }
  }
}

template <bool D3>
__global__ void k_frame_resid(FrameDev f, double* __restrict__ Re) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= f.nele) return;
  element_resid<D3>(f, e, Re);
}

__global__ void k_frame_tangent(FrameDev f, double* __restrict__ Ke) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= f.nele) return;
  element_tangent<false>(f, e, Ke);
}

// The 3D tangent (element_tangent's sums, term by term), 16 lanes per
// element: lanes 0 .. 5 a column each of the basic stiffness over the
// sections, lanes 0 .. 11 a column each of the local and the global one,
// handed on through LDS.  Bound by latency: loads, then three short chains.
// (One thread per element, its matrix rotated in place in global memory:
// 104 elements 21 us; now 5.1.)
__global__ __launch_bounds__(256) void k_frame_tangent3(FrameDev f, double* __restrict__ Ke) {
  __shared__ double skb[16][36];
  __shared__ double skl[16][144];
  const int t = threadIdx.x & 15, le = threadIdx.x >> 4, e = blockIdx.x * 16 + le;
  const bool on = e < f.nele;
  const double* g = f.geo + (long long)(on ? e : 0) * 10;
  const double oneOverL = 1.0 / g[0];
  const long long n = f.nsec;
  const int cb = t < 6 ? t : 5, j = (cb + 1) >> 1;  // section stiffness column
  double kb[6];
#pragma unroll
  for (int i = 0; i < 6; i++) kb[i] = 0.0;
#pragma unroll 5
  for (int i = 0; i < f.nip; i++) {
    const long long sec = (long long)(on ? e : 0) * f.nip + i;
    const double xi6 = 6.0 * (0.5 * (1.0 + gl5_pt(i)));
    const double wti = (gl5_wt(i) * 0.5) * oneOverL;
    const double fc = j == 0 || j == 3 ? 1.0 : (cb & 1) ? xi6 - 4.0 : xi6 - 2.0;
    double ka[4];
#pragma unroll
    for (int k = 0; k < 4; k++) ka[k] = fc * (f.ks[(long long)(j * 4 + k) * n + sec] * wti);
    kb[0] += ka[0];
    kb[1] += (xi6 - 4.0) * ka[1];
    kb[2] += (xi6 - 2.0) * ka[1];
    kb[3] += (xi6 - 4.0) * ka[2];
    kb[4] += (xi6 - 2.0) * ka[2];
    kb[5] += ka[3];
  }
  if (t < 6)
#pragma unroll
    for (int i = 0; i < 6; i++) skb[le][i * 6 + t] = kb[i];
  __syncthreads();
  // column m of kb T, then of T^T kb T: every column of T takes one column
  // of kb or two
  const int m = t < 12 ? t : 11, m6 = m % 6;
  const int c0 = m6 == 0 ? 0 : m6 == 1 ? 1 : m6 == 2 ? 3 : m6 == 3 ? 5 : m6 == 4 ? (m < 6 ? 3 : 4) : (m < 6 ? 1 : 2);
  const int c1 = m6 == 1 ? 2 : m6 == 2 ? 4 : -1;
  const double sc = m6 == 1 ? (m < 6 ? oneOverL : -oneOverL)
                  : m6 == 2 ? (m < 6 ? -oneOverL : oneOverL)
                  : m6 == 0 || m6 == 3 ? (m < 6 ? -1.0 : 1.0)
                                       : 1.0;
  double w[6];
#pragma unroll
  for (int i = 0; i < 6; i++) {
    const double a = skb[le][i * 6 + c0], b = skb[le][i * 6 + (c1 < 0 ? c0 : c1)];
    w[i] = sc * (c1 < 0 ? a : a + b);
  }
  double kl[12];
  kl[0] = -w[0];
  kl[1] = oneOverL * (w[1] + w[2]);
  kl[2] = -oneOverL * (w[3] + w[4]);
  kl[3] = -w[5];
  kl[4] = w[3];
  kl[5] = w[1];
  kl[6] = w[0];
  kl[7] = -kl[1];
  kl[8] = -kl[2];
  kl[9] = w[5];
  kl[10] = w[4];
  kl[11] = w[2];
  if (t < 12)
#pragma unroll
    for (int r = 0; r < 12; r++) skl[le][r * 12 + m] = kl[r];
  __syncthreads();
  // the columns, then the rows, rotated block by block
  const double* R = g + 1;
  const int b3 = 3 * (m / 3), c = m - b3;
  const double r0 = R[c], r1 = R[3 + c], r2 = R[6 + c];
  double x[12];
#pragma unroll
  for (int r = 0; r < 12; r++) {
    const double* row = skl[le] + r * 12 + b3;
    x[r] = row[0] * r0 + row[1] * r1 + row[2] * r2;
  }
  if (!on || t >= 12) return;
  double* K = Ke + (long long)e * 144 + m;
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int q = 0; q < 3; q++)
      K[(3 * b + q) * 12] = R[q] * x[3 * b] + R[3 + q] * x[3 * b + 1] + R[6 + q] * x[3 * b + 2];
}

__global__ void k_copy_d(long long n, const double* __restrict__ a, double* __restrict__ b) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}
__global__ void k_copy_i(long long n, const int* __restrict__ a, int* __restrict__ b) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

void launch_frame_update(hipStream_t s, const FrameDev& f, bool d3, const double* U, int* err) {
  (void)err;
  if (f.nsec <= 0) return;
  if (f.rsec) {
    const dim3 g(ceil_div(f.nrw, 4)), b(256);
    if (f.rw == 20) {
      if (d3) hipLaunchKernelGGL(k_frame_update_rows20<true>, g, b, 0, s, f, U);
      else hipLaunchKernelGGL(k_frame_update_rows20<false>, g, b, 0, s, f, U);
    } else {
      if (d3) hipLaunchKernelGGL(k_frame_update_rows<true>, g, b, 0, s, f, U);
      else hipLaunchKernelGGL(k_frame_update_rows<false>, g, b, 0, s, f, U);
    }
    return;
  }
  const dim3 g(ceil_div(f.nsec, 4)), b(256);
  if (d3) hipLaunchKernelGGL(k_frame_update<true>, g, b, 0, s, f, U);
  else hipLaunchKernelGGL(k_frame_update<false>, g, b, 0, s, f, U);
}
void launch_frame_start(hipStream_t s, const FrameDev& f) {
  if (f.nsec > 0) hipLaunchKernelGGL(k_frame_start, dim3(ceil_div(f.nsec, 4)), dim3(256), 0, s, f);
}
void launch_frame_revert(hipStream_t s, const FrameDev& f, bool d3) {
  if (f.nsec <= 0) return;
  const dim3 g(ceil_div(f.nsec, 4)), b(256);
  if (d3) hipLaunchKernelGGL(k_frame_revert<true>, g, b, 0, s, f);
  else hipLaunchKernelGGL(k_frame_revert<false>, g, b, 0, s, f);
}
void launch_frame_resid(hipStream_t s, const FrameDev& f, bool d3, double* Re) {
  if (f.nele <= 0) return;
  const dim3 g(ceil_div(f.nele, 128)), b(128);
  if (d3) hipLaunchKernelGGL(k_frame_resid<true>, g, b, 0, s, f, Re);
  else hipLaunchKernelGGL(k_frame_resid<false>, g, b, 0, s, f, Re);
}
void launch_frame_tangent(hipStream_t s, const FrameDev& f, bool d3, double* Ke) {
  if (f.nele <= 0) return;
  if (d3) hipLaunchKernelGGL(k_frame_tangent3, dim3(ceil_div(f.nele, 16)), dim3(256), 0, s, f, Ke);
  else hipLaunchKernelGGL(k_frame_tangent, dim3(ceil_div(f.nele, 64)), dim3(64), 0, s, f, Ke);
}
void launch_copy_d(hipStream_t s, long long n, const double* a, double* b) {
  if (n > 0) hipLaunchKernelGGL(k_copy_d, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, a, b);
}
void launch_copy_i(hipStream_t s, long long n, const int* a, int* b) {
  if (n > 0) hipLaunchKernelGGL(k_copy_i, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, a, b);
}

}  // namespace xg
