// mprgp_general.h -- the one-workgroup main loop of the coupled-row solve
// (mprgp_general_dev.hip), as mprgp_general.cpp drives it.
#pragma once
#include "mprgp_host.h"

namespace mprgp {

// Rows of the largest component (rows that share nodes) the one-workgroup loop
// takes: a vertex-triangle contact row and the plane rows of its four nodes
// are five.  A component's QP runs in one wavefront's registers, its block of
// J J^T one entry a lane.
constexpr int kGenBlock = 6;
// Nodes of the largest system: the vector a product gathers from is 24 bytes
// a node of the 64 KB a kernel declares.  There the loop can still be the
// faster one (a beam of 2,499 nodes, 2,511 rows, 271 ms against 570 ms from
// the host over 1,001 iterations), but its products with A, on one CU, grow
// with the matrix.
constexpr int kGenMaxNodes = 2600;
constexpr int kGenMaxRows = 16384;  // some two rows per entry of the largest vector
// What the one-workgroup loop gains on the host-driven one, microseconds an
// iteration: the launches and waits it saves, and about 0.07 for a row that
// shares nodes with no other (three QPs on the host); less the time one CU
// takes for the vectors, the matrix (its load path) and the components of
// several rows (a wavefront each, 16 at a time; the host factors a block in
// less than a wavefront does).  The loop is taken where the estimate is
// positive.  Fitted low to 360 pairs of both loops' times (100 to 2,600 nodes,
// 3 to 300 blocks a row, 0 to 512 components of 1 to 6 rows, none to all of
// their rows active, CG and expansion steps), so that none of those estimated
// positive was slower than from the host.  2,600 nodes, host / one workgroup,
// 3 blocks a row: 16 pairs of rows 202 / 107 us, 256 pairs 313 / 339, 512
// components of six 800 / 1,473; 27 blocks a row, 8 pairs 210 / 242.  A beam
// of 525 nodes with 525 ground rows and 12 contacts 344 / 105.
constexpr double kGenGain = 145.0, kGenRowGain = 0.07, kGenNodeCost = 0.03, kGenSlotCost = 0.0019;
constexpr double kGenCompCost1 = 0.1, kGenCompCost2 = 0.0175;  // k rows: 0.1 k + 0.0175 k^2
// Iterations per launch, so that no launch runs long.
constexpr int kGenChunk = 256;

struct GenState {
  int in_cg;  // the launch ended between two steps of the CG loop, else at the outer loop's head
  int iteration, num_cg, num_exp, num_prop;
  int prop, y_set, ax_set, done, fail;
  double residual, alpha, fx, fy;
};

struct GenArgs {
  int n, m, n_nodes, n_slices;
  const int *sl_off, *col;
  const double *val, *dinv, *b;
  double *x, *g, *p, *z, *phi, *beta, *y, *ap, *t, *t2, *t3, *ax;
  const int *jp, *jc, *tp, *tc;
  const double *jv, *tv, *c;
  unsigned char *face;                  // per row, as the last face decision left it
  double *j1, *j2, *lam, *lam2, *part;  // m, m, m, m; 8 per 256 entries
  // components of several rows: row numbers (-1: none) and J J^T, padded to
  // kGenBlock; components of one row
  int n_big, n_one;
  const int *big_row, *one_row;
  const double *big_g, *one_g;
  double alpha_bar, tol;
  int max_it, pre, chunk;
  GenState *st;
};
hipError_t launch_general_loop(hipStream_t s, const GenArgs *args);  // args in device memory

}  // namespace mprgp
