// Launchers of the tiled sparse factorisation (xg_tiles.hip).
#pragma once
#include <vector>

#include "xg_common.h"

namespace xg {

// Device arrays of a TilePlan (xg_tileplan.h)
struct TileView {
  int nt = 0;
  const int* pos = nullptr;     // position of each equation
  const int* ipos = nullptr;    // equation at each position, -1 on padding
  const int* wid = nullptr;
  const int* colptr = nullptr;
  const int* row = nullptr;
  const int* uptgt = nullptr;
  const int* upsrc = nullptr;
  const int* srcg = nullptr;
  const int* srca = nullptr;
  const int* srck = nullptr;
  const int* fwrow = nullptr;
  const int* fwsrc = nullptr;
  const int* fwg = nullptr;
  const int* fwk = nullptr;
  const int* bwcol = nullptr;
  const int* bwsrc = nullptr;
  const int* bwg = nullptr;
  const int* bwr = nullptr;
  const int4* task = nullptr;   // panel tasks {column, first row tile, row tiles}
};
// Launch ranges, by level
struct TileHost {
  long long tiles = 0;
  std::vector<int> panptr, upptr, fwptr, bwptr;
};

// PCG state of one or two right-hand sides solved side by side
struct TileRhs {
  const double* b;
  double *x, *r, *z, *p, *q;
  int warm;  // x holds a guess and q = A x
};
struct TileScal {
  double bb, rr, rz;
  int conv, iters, fail, pad;
};
struct TilePcg {
  TileRhs v[2];
  TileScal* S;
};

void tiles_factor(hipStream_t s, int n, const TileView& V, const TileHost& H, const int* rowptr, const int* colind,
                  const double* vals, double* A, double* G, int* bad);
// x = (L D L^T)^-1 y for nrhs = 1 or 2 vectors of 64 * nt doubles each, in
// the plan's positions; Y is overwritten
void tiles_sweeps(hipStream_t s, const TileView& V, const TileHost& H, int nrhs, const double* G, double* Y, double* X);
void tiles_in(hipStream_t s, const TileView& V, const double* v, double* y);
void tiles_out(hipStream_t s, int n, const TileView& V, const double* x, double* v);
void tiles_pcg_start(hipStream_t s, int n, int nrhs, const TilePcg& P, double tol2);
void tiles_pcg_dir(hipStream_t s, int n, int nrhs, const TilePcg& P);
void tiles_pcg_step(hipStream_t s, int n, int nrhs, const TilePcg& P, double tol2);

}  // namespace xg
