// Arguments of the pair-lattice kernel (gdx_lattice.hip).
#pragma once
#include "gdx_internal.h"

namespace gdx {

// one part's owned node box
struct LatPart {
  int lo[3], n[3];
  long long base;  // its first row table entry
};

// a row of the global lattice
struct LatRow {
  long long off;       // byte offset of its first value
  int meta;            // pattern id << 9 | has Dirichlet neighbours << 8 | row length (0: no row)
  int bidx;            // its entry of b, -1: no row
};

struct LatArgs {
  int nn[3], ncell[3];  // lattice nodes and cells per direction
  int lo[3], hi[3];     // nodes that may hold rows
  int nt[3];            // tiles
  int pn[3];            // extents of the row table (whole tiles)
  const LatRow *rows;   // on the lattice
  const double *W;  // kappa at the points, or per cell; nullptr: constant
  const uint16_t *delta;  // per pattern: offset in U of every position of the row
  double *values, *b;
  bool source;  // b holds the source integrals already (f varies); else f = fconst
  double kconst, fconst;
  double x0[3], hK[3], dir_coef[4];
  double G[3][6][3], M[3][6][3];  // 1D factors [direction][kind of pair][point]
  double V[3][3][3], Sv[3][3];    // source weights [direction][local node][point] and their sums
};

}  // namespace gdx
