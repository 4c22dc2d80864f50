// Batched ensemble of 2D frame models on gfx950.
//
// A step is one predictor, maxit Newton iterations and one commit; every
// launch covers the whole ensemble:
//   k_ens_predict   -- Newmark::newStep (Newmark.cpp:105-170): predictor and
//                      time advance, a workgroup per model.
//   k_ens_fibers    -- Domain::update: the fibers and sections of every model
//                      still iterating, wavefront items dealt over the whole
//                      chip.
//   k_ens_unbalance -- element forces, ground acceleration (PathSeries),
//                      transient unbalance, CTestNormDispIncr / NormUnbalance,
//                      a workgroup per model.
//   k_ens_iterate   -- the solve of one NewtonRaphson iteration
//                      (NewtonRaphson.cpp:160-215) for every model still
//                      iterating, a workgroup per model: element tangents,
//                      banded assembly of c1 K + c2 C + c3 M in element order
//                      (in LDS where it fits), banded L D L^T and solve by one
//                      wavefront for bands up to 24, Newmark::update.
//   k_ens_commit    -- Domain::commit of converged models (nodal state; the
//                      fiber pools commit by exchanging the committed and
//                      trial pool pointers); revert of models whose Newton
//                      failed (they stop, as analyze returns < 0).
// The fibers carry the work (77% of it) and the models differ tenfold in
// size: with a whole iteration in one workgroup per model, a step of 300
// frames of 3 to 20 stories waited for its largest one (11.4 ms a step; now
// 5.0, of which the fiber launches at 4.7 TB/s take 2.4; 1,200 frames 22.3 and
// 17.1, 20 frames 6.7 and 1.5).  Once no model iterates, the fiber launches left in the step read
// one counter and end.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "xg_ensemble.h"
#include "xg_frame_impl.h"

namespace xg {

template <int NT>
__device__ __forceinline__ double block_sum_t(double v, double* sh) {
  // wavefront butterfly (every lane ends with the same bits: each step adds
  // the same two operands in either order), then the NT / 64 wave sums in
  // wave order: one barrier pair instead of a log2(NT)-level LDS tree
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if constexpr (NT == 64) {
    return v;
  } else {
    const int t = threadIdx.x;
    if ((t & 63) == 0) sh[t >> 6] = v;
    __syncthreads();
    double r = sh[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) r += sh[w];
    __syncthreads();
    return r;
  }
}

__device__ __forceinline__ double path_accel(const EnsDev& E, int m, double t) {
  const int n = E.gm_n[m];
  const double h = E.gm_dt[m];
  if (n <= 0 || !(h > 0.0) || t < 0.0) return 0.0;
  const double incr = t / h;
  const int i1 = (int)floor(incr);
  const int i2 = i1 + 1;
  if (i2 >= n) return 0.0;
  const double* g = E.gm + E.gm_off[m];
  const double v1 = g[i1], v2 = g[i2];
  return E.gm_fac[m] * (v1 + (v2 - v1) * (incr - i1));
}

// Element forces and transient unbalance of model m (all threads of the
// block)
template <int NT>
__device__ void model_unbalance(const EnsDev& E, int m, double ag) {
  const int tid = threadIdx.x;
  for (int e = E.ele_off[m] + tid; e < E.ele_off[m + 1]; e += NT) element_resid<false>(E.f, e, E.Re);
  __syncthreads();
  const double alphaM = E.alphaM[m];
  for (int a = E.eq_off[m] + tid; a < E.eq_off[m + 1]; a += NT) {
    double acc = 0.0;
    for (int j = E.rhs_ptr[a]; j < E.rhs_ptr[a + 1]; j++) acc += -E.Re[E.rhs_idx[j]];
    double u = 0.0;
    const double mm = E.M[a];
    if (mm != 0.0) {
      const int d = E.eq2dof[a];
      u += -(mm * E.R[a]) * ag;
      u += -mm * E.A[d];
      if (alphaM != 0.0) u += -alphaM * mm * E.V[d];
    }
    E.B[a] = acc + u;
  }
  __syncthreads();
}

// The fiber update of every running model (First: of a step's predictor;
// else of the models still iterating), one wavefront item (three sections
// in 20-lane rows, or one section) at a time.
template <bool First>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_ens_fibers(EnsDev E) {
  __shared__ double red[4 * 5 * 64];
  if (*E.active == 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long step = (long long)gridDim.x * 4;
  for (long long w = (long long)blockIdx.x * 4 + wave; w < E.nitem; w += step) {
    if (E.status[E.item_model[w]] != 0) continue;
    if (E.rows) section_rows<false, 20, First>(E.f, w, lane, E.U, red + wave * 5 * 64);
    else section_update<false, First>(E.f, w, lane, E.U);
  }
}

__device__ __forceinline__ double readlane_d(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// 1/a: the hardware estimate and two Newton steps
__device__ __forceinline__ double rcp_d(double a) {
  double y = __builtin_amdgcn_rcp(a);
  y = fma(y, fma(-a, y, 1.0), y);
  return fma(y, fma(-a, y, 1.0), y);
}

// The value again, as one the compiler cannot trace: what is computed from
// it stays where it is used (the lane's addresses and masks of all pivots of
// a pass, taken out of the loop over passes, filled 3.4 KB of scratch)
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// One pivot of wave_band_solve, j = j0 + P.
template <int P, int BW, int WIN>
__device__ __forceinline__ void band_pivot(double* Lb, double* zb, int ld, int bw, int n, int j, int l,
                                           double (&w)[WIN], double& y, int& bad) {
  constexpr int M = WIN - 1;
  const double d = readlane_d(w[P], P), yj = readlane_d(y, P);
  if (!(d > 0.0)) bad = 1;
  const double inv = rcp_d(d), u = w[P] * inv;
  const int dl = (opaque(l) - P) & M;  // the lane's row below the pivot
  if (j < n && dl <= bw) Lb[j * ld + dl] = u;
  if (j < n && dl == 0) zb[j] = yj * inv;
  y = fma(-u, yj, y);
#pragma unroll
  for (int c = 1; c <= BW; c++) w[(P + c) & M] = fma(-u, readlane_d(w[P], (P + c) & M), w[(P + c) & M]);
  // every update now: left to itself the compiler puts a column's updates
  // off to its own pivot, with all the broadcasts in between spilled
#pragma unroll
  for (int c = 1; c <= BW; c++) asm volatile("" : "+v"(w[(P + c) & M]));
}
// One step of the backward sweep, i = i0 + P (u: the lane's entry of row i)
template <int P>
__device__ __forceinline__ void band_back(double u, double& z) {
  z = fma(-u, readlane_d(z, P), z);
}

template <int BW, int WIN, int B0, int... Ps>
__device__ __forceinline__ void band_batch(std::integer_sequence<int, Ps...>, double* Lb, double* zb, int ld, int bw,
                                           int n, int j0, int l, double (&w)[WIN], double& y, int& bad) {
  (band_pivot<B0 + Ps, BW, WIN>(Lb, zb, ld, bw, n, j0 + B0 + Ps, l, w, y, bad), ...);
}
template <int BW, int WIN, int BATCH, int... Bs, class Load>
__device__ __forceinline__ void band_pass(std::integer_sequence<int, Bs...>, double* Lb, double* zb, int ld, int bw,
                                          int n, int j0, int l, double (&w)[WIN], double& y, int& bad, Load load) {
  auto one = [&](auto bi) __attribute__((always_inline)) {
    constexpr int B0 = decltype(bi)::value * BATCH;
    band_batch<BW, WIN, B0>(std::make_integer_sequence<int, BATCH>{}, Lb, zb, ld, bw, n, j0, l, w, y, bad);
    if (l >= B0 && l < B0 + BATCH) load(j0 + WIN + l);
  };
  (one(std::integral_constant<int, Bs>{}), ...);
}
template <int WIN, int B0, int... Ps>
__device__ __forceinline__ void band_back_batch(std::integer_sequence<int, Ps...>, const double (&u)[sizeof...(Ps)],
                                                double& z) {
  constexpr int N = sizeof...(Ps);
  (band_back<B0 + N - 1 - Ps>(u[N - 1 - Ps], z), ...);
}
template <int WIN, int BATCH, int... Bs, class Z>
__device__ __forceinline__ void band_back_pass(std::integer_sequence<int, Bs...>, const double* Lb, int ld, int bw,
                                               int n, int i0, int l, double& z, Z z_at, double* x) {
  auto one = [&](auto bi) __attribute__((always_inline)) {
    constexpr int B0 = (WIN / BATCH - 1 - decltype(bi)::value) * BATCH;
    double u[BATCH];
    const int lo = opaque(l);
#pragma unroll
    for (int q = 0; q < BATCH; q++) {
      const int i = i0 + B0 + q, dl = (B0 + q - lo) & (WIN - 1), r = i - dl;
      const bool held = i < n && dl >= 1 && dl <= bw && r >= 0;
      const double v = Lb[held ? r * ld + dl : 0];
      u[q] = held ? v : 0.0;
    }
    band_back_batch<WIN, B0>(std::make_integer_sequence<int, BATCH>{}, u, z);
    __builtin_amdgcn_sched_barrier(0);
    if (l >= B0 && l < B0 + BATCH) {
      const int r = i0 + l;
      if (r < n) x[r] = z;
      z = z_at(r - WIN);
    }
  };
  (one(std::integral_constant<int, Bs>{}), ...);
}

// Banded L D L^T = A (L unit lower) and solve, by one wavefront (no
// barriers).  A is symmetric positive definite with half bandwidth bw <= BW,
// stored by rows: A(r, c) = Lb[r*ld + c - r + bw] for r - bw <= c <= r.
// Lane l (and l + WIN, ...) holds row r = l mod WIN of the active window, its
// column c in w[c mod WIN]: no value moves between lanes, every register
// index is a constant (WIN pivots to a pass), and after BATCH pivots their
// lanes take the rows WIN further down.  Column j of L overwrites band row j.
// zb: n doubles; x receives the solution.  Returns nonzero if a pivot is not
// positive.  (Shifting the window a row per pivot, with Cholesky's square
// root and divisions on the chain: 20 frames 2.7 ms a step, now 1.5.)
template <int BW, int WIN, int BATCH>
__device__ __forceinline__ int wave_band_solve(double* Lb, double* zb, int ld, int bw, int n,
                                               const double* __restrict__ b, double* x) {
  static_assert(BW + BATCH <= WIN && WIN % BATCH == 0, "window");
  constexpr int M = WIN - 1;
  const int l = threadIdx.x & M;
  double w[WIN], y = 0.0;
  auto load = [&](int row) __attribute__((always_inline)) {
    const int r = opaque(row), at = r * ld + bw;
    const bool in = r < n, pad = !in;
#pragma unroll
    for (int m = 0; m < WIN; m++) {
      const int back = (r - m) & M;  // column r - back
      const bool held = in && back <= bw;
      const double v = Lb[held ? at - back : 0];
      w[m] = held ? v : pad && back == 0 ? 1.0 : 0.0;
    }
    y = in ? b[r] : 0.0;
  };
  load(l);
  int bad = 0;
#pragma unroll 1
  for (int j0 = 0; j0 < n; j0 += WIN) {
    band_pass<BW, WIN, BATCH>(std::make_integer_sequence<int, WIN / BATCH>{}, Lb, zb, ld, bw, n, j0, l, w, y, bad, load);
  }
  // backward: x_i = z_i - sum_k L(i + k, i) x_{i+k}; lane l holds the pending
  // value of row r = l mod WIN, row i of L comes one entry to a lane
  const int top = (n + WIN - 1) / WIN * WIN;
  auto z_at = [&](int r) { return r >= 0 && r < n ? zb[r] : 0.0; };
  double z = z_at(top - WIN + l);
#pragma unroll 1
  for (int i0 = top - WIN; i0 >= 0; i0 -= WIN)
    band_back_pass<WIN, BATCH>(std::make_integer_sequence<int, WIN / BATCH>{}, Lb, ld, bw, n, i0, l, z, z_at, x);
  return bad;
}

template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_ens_predict(EnsDev E) {
  for (int k = blockIdx.x; k < E.nmodel; k += gridDim.x) {
    const int m = E.order[k];
    if (E.status[m] <= -2) continue;  // stopped after a failed step
    const int tid = threadIdx.x;
    const double g = E.gamma, b = E.beta, h = E.dt;
    const double a1 = (1.0 - g / b), a2 = h * (1.0 - 0.5 * g / b), a3 = -1.0 / (b * h), a4 = 1.0 - 0.5 / b;
    const int d0 = E.node_off[m] * E.ndf, d1 = E.node_off[m + 1] * E.ndf;
    for (int d = d0 + tid; d < d1; d += NT) {
      if (E.eqmap[d] < 0) continue;
      E.U[d] = E.Uc[d];
      E.V[d] = E.Vc[d] * a1 + E.Ac[d] * a2;
      E.A[d] = E.Ac[d] * a4 + E.Vc[d] * a3;
    }
    if (tid == 0) {
      E.iter[m] = 0;
      E.status[m] = 0;
      atomicAdd(E.active, 1);
    }
  }
}

// Unbalance of the models still iterating; after the predictor (First) that
// is all, after an iteration the convergence test follows.
template <int NT, bool First>
__device__ __forceinline__ void ens_unbalance(const EnsDev& E) {
  __shared__ double sh[NT];
  for (int k = blockIdx.x; k < E.nmodel; k += gridDim.x) {
    const int m = E.order[k];
    if (E.status[m] != 0) continue;
    const int tid = threadIdx.x;
    // E.time holds the committed time; the trial time is E.time + dt
    // (Newmark.cpp newStep: time += deltaT), formed the same way everywhere
    model_unbalance<NT>(E, m, path_accel(E, m, E.time[m] + E.dt));
    if (First) continue;
    double v = 0.0;
    const double* w = E.test_kind == 1 ? E.B : E.X;
    for (int a = E.eq_off[m] + tid; a < E.eq_off[m + 1]; a += NT) v += w[a] * w[a];
    const double norm = sqrt(block_sum_t<NT>(v, sh));
    if (tid == 0) {
      const int it = E.iter[m] + 1;
      E.iter[m] = it;
      E.norm[m] = norm;
      E.newton_count[m] += 1;
      if (norm <= E.tol) E.status[m] = 1;
      else if (it >= E.maxit) E.status[m] = -1;
      if (norm <= E.tol || it >= E.maxit) atomicAdd(E.active, -1);
    }
    __syncthreads();
  }
}
template <int NT>
__global__ __launch_bounds__(NT) void k_ens_unbalance_first(EnsDev E) {
  ens_unbalance<NT, true>(E);
}
template <int NT>
__global__ __launch_bounds__(NT) void k_ens_unbalance(EnsDev E) {
  ens_unbalance<NT, false>(E);
}

template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_ens_iterate(EnsDev E) {
  extern __shared__ double lband[];
  __shared__ int s_bad;
  for (int k = blockIdx.x; k < E.nmodel; k += gridDim.x) {
    const int m = E.order[k];
    if (E.status[m] != 0) continue;
    const int tid = threadIdx.x;
    const int eq0 = E.eq_off[m], n = E.eq_off[m + 1] - eq0;
    const int bw = E.bw[m], ld = bw + 1;
    const long long bo = E.band_off[m];
    double* L = E.band + bo;
    const double g = E.gamma, b = E.beta, h = E.dt;
    const double c2 = g / (b * h), c3 = 1.0 / (b * h * h);
    const double mc = c3 + c2 * E.alphaM[m];
    // ---- tangent: element K, then c1 K + c2 C + c3 M into the band ----
    for (int e = E.ele_off[m] + tid; e < E.ele_off[m + 1]; e += NT) element_tangent<false>(E.f, e, E.Ke);
    if (tid == 0) s_bad = 0;
    double* x = E.X + eq0;
    const double* rhs = E.B + eq0;
    const bool lds = bw <= 24 && (long long)n * (ld + 1) <= E.lds_doubles;
    auto assemble = [&](double* T) __attribute__((always_inline)) {
      for (long long i = tid; i < (long long)n * ld; i += NT) T[i] = 0.0;
      __syncthreads();
      for (int q = E.bent_off[m] + tid; q < E.bent_off[m + 1]; q += NT) {
        double acc = 0.0;
        for (int j = E.bent_ptr[q]; j < E.bent_ptr[q + 1]; j++) acc += E.Ke[E.bent_idx[j]];
        T[E.bent_pos[q] - bo] = acc;
      }
      __syncthreads();
      for (int a = tid; a < n; a += NT) {
        const double mm = E.M[eq0 + a];
        if (mm != 0.0) T[(long long)a * ld + bw] += mc * mm;
      }
      __syncthreads();
    };
    auto solve = [&](double* T, double* zb) __attribute__((always_inline)) {
      if (tid < 64) {
        int bad;
        if (bw <= 8) bad = wave_band_solve<8, 16, 8>(T, zb, ld, bw, n, rhs, x);
        else if (bw <= 16) bad = wave_band_solve<16, 32, 16>(T, zb, ld, bw, n, rhs, x);
        else bad = wave_band_solve<24, 32, 8>(T, zb, ld, bw, n, rhs, x);
        if (tid == 0 && bad) s_bad = 1;
      }
      __syncthreads();
    };
    if (lds) {
      assemble(lband);
      solve(lband, lband + (long long)n * ld);
    } else {
      assemble(L);
      if (bw <= 24) solve(L, x);  // the forward values pass through x itself
      // ---- wide bands: left-looking banded Cholesky by columns ----
      for (int j = 0; bw > 24 && j < n; j++) {
        if (tid == 0) {
          double s = L[(long long)j * ld + bw];
          const int k0 = j - bw > 0 ? j - bw : 0;
          for (int kk = k0; kk < j; kk++) {
            const double v = L[(long long)j * ld + (kk - j + bw)];
            s -= v * v;
          }
          if (!(s > 0.0)) s_bad = 1;
          L[(long long)j * ld + bw] = sqrt(s > 0.0 ? s : 1.0);
        }
        __syncthreads();
        const double djj = L[(long long)j * ld + bw];
        for (int r = tid; r < bw; r += NT) {
          const int i = j + 1 + r;
          if (i >= n) break;
          double s = L[(long long)i * ld + (j - i + bw)];
          const int k0 = i - bw > 0 ? i - bw : 0;
          for (int kk = k0; kk < j; kk++)
            s -= L[(long long)i * ld + (kk - i + bw)] * L[(long long)j * ld + (kk - j + bw)];
          L[(long long)i * ld + (j - i + bw)] = s / djj;
        }
        __syncthreads();
      }
      if (bw > 24 && tid == 0) {
        for (int i = 0; i < n; i++) {
          double s = rhs[i];
          const int k0 = i - bw > 0 ? i - bw : 0;
          for (int kk = k0; kk < i; kk++) s -= L[(long long)i * ld + (kk - i + bw)] * x[kk];
          x[i] = s / L[(long long)i * ld + bw];
        }
        for (int i = n - 1; i >= 0; i--) {
          double s = x[i];
          const int k1 = i + bw < n - 1 ? i + bw : n - 1;
          for (int kk = i + 1; kk <= k1; kk++) s -= L[(long long)kk * ld + (i - kk + bw)] * x[kk];
          x[i] = s / L[(long long)i * ld + bw];
        }
      }
      __syncthreads();
    }
    if (s_bad) {
      if (tid == 0) {
        E.status[m] = -1;  // BadLinearSolve
        atomicAdd(E.active, -1);
      }
      __syncthreads();
      continue;
    }
    // ---- Newmark::update ----
    const int d0 = E.node_off[m] * E.ndf, d1 = E.node_off[m + 1] * E.ndf;
    for (int d = d0 + tid; d < d1; d += NT) {
      const int a = E.eqmap[d];
      if (a < 0) continue;
      const double du = E.X[a];
      E.U[d] += du;
      E.V[d] += c2 * du;
      E.A[d] += c3 * du;
    }
    __syncthreads();
  }
}

// commit converged models; revert (and stop) models whose step failed
template <int NT>
__global__ __launch_bounds__(NT) void k_ens_commit(EnsDev E) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *E.active = 0;
  for (int k = blockIdx.x; k < E.nmodel; k += gridDim.x) {
    const int m = E.order[k];
    const int st = E.status[m];
    if (st <= -2) continue;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int d0 = E.node_off[m] * E.ndf, d1 = E.node_off[m + 1] * E.ndf;
    const long long s0 = (long long)E.ele_off[m] * E.f.nip, s1 = (long long)E.ele_off[m + 1] * E.f.nip;
    if (st == 1) {
      if (tid == 0) E.time[m] += E.dt;
      for (int d = d0 + tid; d < d1; d += NT) {
        E.Uc[d] = E.U[d];
        E.Vc[d] = E.V[d];
        E.Ac[d] = E.A[d];
      }
      // the fiber state commits by the host exchanging the committed and
      // trial pools after this kernel (Ensemble::flip)
    } else {
      // failed (or never converged within the launched iterations):
      // Domain::revertToLastCommit and stop this model
      for (int d = d0 + tid; d < d1; d += NT) {
        E.U[d] = E.Uc[d];
        E.V[d] = E.Vc[d];
        E.A[d] = E.Ac[d];
      }
      for (long long sec = s0 + wave; sec < s1; sec += NT / 64) section_revert<false>(E.f, sec, lane);
      __syncthreads();
      if (tid == 0) E.status[m] = -2;
    }
    __syncthreads();
  }
}

#define XG_ENS_DISPATCH(KERNEL, LDS, ...)                                                                 \
  switch (block) {                                                                                     \
    case 128: hipLaunchKernelGGL(KERNEL<128>, dim3(grid), dim3(128), LDS, s, __VA_ARGS__); break;       \
    case 512: hipLaunchKernelGGL(KERNEL<512>, dim3(grid), dim3(512), LDS, s, __VA_ARGS__); break;       \
    default: hipLaunchKernelGGL(KERNEL<256>, dim3(grid), dim3(256), LDS, s, __VA_ARGS__); break;        \
  }

// enough workgroups to fill the chip's wavefront slots once over
static dim3 fiber_grid(const EnsDev& E) {
  return dim3((unsigned)std::max<long long>(1, std::min<long long>((E.nitem + 3) / 4, 2048)));
}
void launch_ens_predict(hipStream_t s, const EnsDev& E, int grid, int block) {
  XG_ENS_DISPATCH(k_ens_predict, 0, E);
  hipLaunchKernelGGL(k_ens_fibers<true>, fiber_grid(E), dim3(256), 0, s, E);
  XG_ENS_DISPATCH(k_ens_unbalance_first, 0, E);
}
void launch_ens_iterate(hipStream_t s, const EnsDev& E, int grid, int block) {
  XG_ENS_DISPATCH(k_ens_iterate, E.lds_doubles * sizeof(double), E);
  hipLaunchKernelGGL(k_ens_fibers<false>, fiber_grid(E), dim3(256), 0, s, E);
  XG_ENS_DISPATCH(k_ens_unbalance, 0, E);
}
void launch_ens_commit(hipStream_t s, const EnsDev& E, int grid, int block) { XG_ENS_DISPATCH(k_ens_commit, 0, E); }

}  // namespace xg
