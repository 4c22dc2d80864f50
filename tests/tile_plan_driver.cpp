// CPU driver for the host code of the tiled sparse factorisation's plan
// (xg_tileplan.h).
//   tile_plan_driver IN OUT: IN: n, nnode, ndf, ndm, nnz (int32), rowptr[n +
//     1], colind[nnz], eq[nnode*ndf] (int32), crd[nnode*ndm], max_tiles,
//     max_flops (double).  OUT: ok, nt, nlev, then each array of the plan as
//     its length and values (int32).
#include <cstdio>
#include <vector>

#include "../xara_amd/csrc/xg_tileplan.h"

template <class T>
static bool rd(FILE* f, std::vector<T>& v, size_t n) {
  v.resize(n);
  return n == 0 || fread(v.data(), sizeof(T), n, f) == n;
}

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  FILE* f = fopen(argv[1], "rb");
  if (!f) return 2;
  std::vector<int> h, rp, ci, eq;
  std::vector<double> crd, lim;
  if (!rd(f, h, 5) || !rd(f, rp, h[0] + 1) || !rd(f, ci, h[4]) || !rd(f, eq, (size_t)h[1] * h[2]) ||
      !rd(f, crd, (size_t)h[1] * h[3]) || !rd(f, lim, 2))
    return 2;
  fclose(f);
  xg::TilePlan P;
  const int ok = xg::tile_plan(h[0], rp, ci, h[1], h[2], h[3], eq, crd, (long long)lim[0], lim[1], P) ? 1 : 0;
  FILE* g = fopen(argv[2], "wb");
  if (!g) return 2;
  const int head[3] = {ok, P.nt, P.nlev};
  fwrite(head, sizeof(int), 3, g);
  if (ok)
    for (auto* v : {&P.pos, &P.wid, &P.colptr, &P.row, &P.lev, &P.levptr, &P.levcol, &P.upptr, &P.uptgt, &P.upsrc,
                    &P.srcg, &P.srca, &P.srck, &P.fwptr, &P.fwrow, &P.fwsrc, &P.fwg, &P.fwk, &P.bwptr, &P.bwcol,
                    &P.bwsrc, &P.bwg, &P.bwr}) {
      const int n = (int)v->size();
      fwrite(&n, sizeof(int), 1, g);
      fwrite(v->data(), sizeof(int), v->size(), g);
    }
  fclose(g);
  return 0;
}
