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

template <bool D3>
__global__ void k_frame_tangent(FrameDev f, double* __restrict__ Ke) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= f.nele) return;
  element_tangent<D3>(f, e, Ke);
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
  const dim3 g(ceil_div(f.nele, 64)), b(64);
  if (d3) hipLaunchKernelGGL(k_frame_tangent<true>, g, b, 0, s, f, Ke);
  else hipLaunchKernelGGL(k_frame_tangent<false>, g, b, 0, s, f, Ke);
}
void launch_copy_d(hipStream_t s, long long n, const double* a, double* b) {
  if (n > 0) hipLaunchKernelGGL(k_copy_d, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, a, b);
}
void launch_copy_i(hipStream_t s, long long n, const int* a, int* b) {
  if (n > 0) hipLaunchKernelGGL(k_copy_i, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, a, b);
}

}  // namespace xg
