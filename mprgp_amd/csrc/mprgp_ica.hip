// mprgp_ica.hip -- the ICA comparator on the device: ICASolver
// (ICASolver.h:287-463; Otaduy et al., "Implicit Contact Handling for
// Deformable Objects", EG 2009), the solver the reference benchmarks MPRGP
// against (ICAFemSolver::forward, MprgpFemSolver.cpp:439-486), for
//     A x = b + J^T lambda,  0 <= lambda  _|_  J x - p >= 0.
//
// A = La + Da + Ua (3x3 diagonal blocks Da; La / Ua the blocks whose node
// comes before / after the row's node in the user's order).  Each iteration:
//     c      = p + J Da^-1 (LaUa x - b)        ica_rows(kOffDiag), J u
//     lambda = projected Gauss-Seidel on B = J Da^-1 J^T from the previous
//              lambda (host: B is m x m and the sweep is serial)
//     rhs    = J^T lambda - Ua x + b           ica_rows(kUpper)
//     x      = one forward block Gauss-Seidel sweep of (Da + La) x = rhs
//     |A x - b - J^T lambda| <= tol stops      ica_rows(kResidual), dot
//
// The sweep is sequential in the user's node order, and it stays so: nodes
// are grouped into dependency levels (a node's level is one more than the
// highest level among the nodes it couples to that come before it), and one
// workgroup runs the levels in order with a barrier between them, x in an
// LDS ring where the levels' reach allows (ica_sweep_ring).  Every node then
// sees exactly the new and old values the sequential sweep gives it, so the
// sweep is the reference's, not a multicolour variant with other iterates.  Each row adds its terms in the order of its blocks (the input's
// column order), singly rounded, as the oracle does.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "mprgp_host.h"

// no fused multiply-adds: each product and sum is rounded once, in the
// oracle's order
#pragma clang fp contract(off)

namespace mprgp {
namespace {

enum IcaRowMode { kOffDiag = 0, kUpper = 1, kResidual = 2 };

// 3x3 inverse (row-major) by the adjugate: inv(i,j) = cof(j,i) / det.
__device__ __forceinline__ void inv3(const double *m, double *inv) {
  const double c00 = m[4] * m[8] - m[5] * m[7];
  const double c01 = m[5] * m[6] - m[3] * m[8];
  const double c02 = m[3] * m[7] - m[4] * m[6];
  const double c10 = m[2] * m[7] - m[1] * m[8];
  const double c11 = m[0] * m[8] - m[2] * m[6];
  const double c12 = m[1] * m[6] - m[0] * m[7];
  const double c20 = m[1] * m[5] - m[2] * m[4];
  const double c21 = m[2] * m[3] - m[0] * m[5];
  const double c22 = m[0] * m[4] - m[1] * m[3];
  const double det = m[0] * c00 + m[1] * c01 + m[2] * c02;
  inv[0] = c00 / det; inv[1] = c10 / det; inv[2] = c20 / det;
  inv[3] = c01 / det; inv[4] = c11 / det; inv[5] = c21 / det;
  inv[6] = c02 / det; inv[7] = c12 / det; inv[8] = c22 / det;
}

// Da^-1 per internal node: the row's block on its own node (padding slots
// also point at the row's node and add zeros).
__global__ void __launch_bounds__(256) ica_dinv(const int *sl_off, const int *col, const double *val, int n_nodes,
                                                double *dinv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_nodes) return;
  const int s = i / kSlice, l = i % kSlice;
  const int b0 = sl_off[s], W = (sl_off[s + 1] - b0) / kSlice;
  double D[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int k = 0; k < W; ++k) {
    if (col[b0 + k * kSlice + l] != i) continue;
    const double *v = val + (size_t)b0 * 9 + (size_t)k * 9 * kSlice + l;
    for (int e = 0; e < 9; ++e) D[e] += v[e * kSlice];
  }
  inv3(D, dinv + 9 * (size_t)i);
}

// Cross-lane: the value of the quad's lane kLane.
template <int kLane>
__device__ __forceinline__ double quad_lane(double v) {
  constexpr int ctrl = kLane | kLane << 2 | kLane << 4 | kLane << 6;
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// One pass over each row's blocks (internal node order, 3 values per node):
//   kOffDiag:  out = Da^-1 (sum over blocks off the node of A x  -  b)
//   kUpper:    out = (jtl - sum over blocks after the node of A x) + b
//   kResidual: out = (A x - b) - jtl
__global__ void __launch_bounds__(256) ica_rows(const int *sl_off, const int *col, const double *val,
                                                const int *perm, const double *x, const double *b,
                                                const double *jtl, const double *dinv, double *out, int n_nodes,
                                                int mode, const int *pos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_nodes) return;
  const int s = i / kSlice, l = i % kSlice;
  const int b0 = sl_off[s], W = (sl_off[s + 1] - b0) / kSlice;
  const int ui = perm[i];
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  for (int k = 0; k < W; ++k) {
    const int c = col[b0 + k * kSlice + l];
    const bool take = mode == kOffDiag ? c != i : (mode == kUpper ? perm[c] > ui : true);
    if (!take) continue;
    const double *v = val + (size_t)b0 * 9 + (size_t)k * 9 * kSlice + l;
    const double x0 = x[3 * (size_t)c], x1 = x[3 * (size_t)c + 1], x2 = x[3 * (size_t)c + 2];
    a0 += v[0 * kSlice] * x0;
    a0 += v[1 * kSlice] * x1;
    a0 += v[2 * kSlice] * x2;
    a1 += v[3 * kSlice] * x0;
    a1 += v[4 * kSlice] * x1;
    a1 += v[5 * kSlice] * x2;
    a2 += v[6 * kSlice] * x0;
    a2 += v[7 * kSlice] * x1;
    a2 += v[8 * kSlice] * x2;
  }
  const size_t r = 3 * (size_t)i;
  if (mode == kOffDiag) {
    const double t0 = a0 - b[r], t1 = a1 - b[r + 1], t2 = a2 - b[r + 2];
    const double *D = dinv + 9 * (size_t)i;
    out[r] = D[0] * t0 + D[1] * t1 + D[2] * t2;
    out[r + 1] = D[3] * t0 + D[4] * t1 + D[5] * t2;
    out[r + 2] = D[6] * t0 + D[7] * t1 + D[8] * t2;
  } else if (mode == kUpper) {
    double *o = out + 3 * (size_t)(pos ? pos[i] : i);  // pos: the sweep's order
    o[0] = (jtl[r] - a0) + b[r];
    o[1] = (jtl[r + 1] - a1) + b[r + 1];
    o[2] = (jtl[r + 2] - a2) + b[r + 2];
  } else {
    out[r] = (a0 - b[r]) - jtl[r];
    out[r + 1] = (a1 - b[r + 1]) - jtl[r + 1];
    out[r + 2] = (a2 - b[r + 2]) - jtl[r + 2];
  }
}

// The lower blocks' values in sweep order, 9 per block (row-major), gathered
// once per call from their SELL slots: a slot's 9 values, for slice base b0
// and block k with slot = b0 + 64 k + l, sit at 9 (b0 + 64 k) + l + 64 e.
__global__ void __launch_bounds__(256) ica_lower_vals(const double *val, const int *lo_slot, int n_lo,
                                                      double *lo_val) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n_lo) return;
  const long long slot = lo_slot[e];
  const double *v = val + (9 * slot - 8 * (slot % kSlice));
#pragma unroll
  for (int k = 0; k < 9; ++k) lo_val[9 * (size_t)e + k] = v[k * kSlice];
}

// The forward block Gauss-Seidel sweep (ICASolver.h:394-404) in one
// workgroup, level by level, one thread per node of a level.  A level's
// nodes depend only on nodes of earlier levels, whose x the barrier after
// each level publishes.  A node's lower blocks (its blocks on nodes before
// it) are listed in sweep order, lo_ptr[t] .. lo_ptr[t + 1] for the
// level-ordered node t, with their values copied in that order (lo_val) and
// their columns; the thread loads them kChunk at a time, every load of a
// chunk issued before the chunk's products, and subtracts v_ab x_b (each
// product rounded once: no contraction in this file) from rhs in block
// order, b = 0, 1, 2, as the sequential sweep does; then x = Da^-1 r.
constexpr int kChunk = 6;
__global__ void __launch_bounds__(512) ica_sweep(const double *lo_val, const int *lo_col, const int *lo_ptr,
                                                 const double *dinv, const double *rhs, double *x,
                                                 const int *lvl_ptr, const int *lvl_node, int n_levels) {
  for (int lv = 0; lv < n_levels; ++lv) {
    const int t1 = lvl_ptr[lv + 1];
    for (int t = lvl_ptr[lv] + (int)threadIdx.x; t < t1; t += (int)blockDim.x) {
      const int i = lvl_node[t], k0 = lo_ptr[t], k1 = lo_ptr[t + 1];
      const size_t r = 3 * (size_t)i;
      double r0 = rhs[r], r1 = rhs[r + 1], r2 = rhs[r + 2];
      const double *D = dinv + 9 * (size_t)i;
      for (int e0 = k0; e0 < k1; e0 += kChunk) {
        double v[kChunk][9], xb[kChunk][3];
#pragma unroll
        for (int u = 0; u < kChunk; ++u) {
          const int e = min(e0 + u, k1 - 1);  // past the node's last block: its last again, not used
          const int c = lo_col[e];
#pragma unroll
          for (int k = 0; k < 9; ++k) v[u][k] = lo_val[9 * (size_t)e + k];
#pragma unroll
          for (int k = 0; k < 3; ++k) xb[u][k] = x[3 * (size_t)c + k];
        }
        asm volatile("" ::: "memory");  // the chunk's loads stay ahead of its products
#pragma unroll
        for (int u = 0; u < kChunk; ++u) {
          if (e0 + u >= k1) break;
          r0 -= v[u][0] * xb[u][0];
          r0 -= v[u][1] * xb[u][1];
          r0 -= v[u][2] * xb[u][2];
          r1 -= v[u][3] * xb[u][0];
          r1 -= v[u][4] * xb[u][1];
          r1 -= v[u][5] * xb[u][2];
          r2 -= v[u][6] * xb[u][0];
          r2 -= v[u][7] * xb[u][1];
          r2 -= v[u][8] * xb[u][2];
        }
      }
      x[r] = D[0] * r0 + D[1] * r1 + D[2] * r2;
      x[r + 1] = D[3] * r0 + D[4] * r1 + D[5] * r2;
      x[r + 2] = D[6] * r0 + D[7] * r1 + D[8] * r2;
    }
    __syncthreads();
  }
}

constexpr int kSweepThreads = 512;

// The same sweep with x kept in the LDS.  The sweep is one CU's work and was
// bound by each level's chain: level bounds, node and block range, columns,
// x, products, the store of x and its acknowledgement before the barrier.
// Here a level's x goes to a ring in the LDS (slot: position in the sweep's
// order modulo kRing), so a level waits for LDS traffic only, and everything
// that does not depend on x is loaded one level ahead and stays in flight
// across the barrier.  Four lanes per node, lane c < 3 for scalar row c: a
// node's kAhead first lower blocks are three values each in registers.  Per
// level the blocks are stored [block][node], so a load is consecutive over
// the lanes.  A scalar row's products are subtracted in the same order as by
// one thread per node.
//   lvl       per level: first position, nodes, first padded block, blocks per
//             node (the most any node of the level has)
//   lo_ring   per padded block, [node][block]: 3 times the ring slot of its
//             column (kAhead are read from a node's first on)
//   lo_val    9 values per padded block
//   lo_cnt    per position: the node's lower blocks
//   dinv, rhs per position; node: the internal node at a position
// Used where every column a level reads is among the kRing positions up to
// the level's end (the caller checks); a level past 128 nodes (four lanes each)
// runs in passes.
// Measured on a beam of 3,402 nodes in 148 levels: an iteration 443 -> 222 us
// (with the wait merged below); what is left per level is the load path of
// one CU, about 35 bytes a cycle.
constexpr int kRing = 6400;  // 150 KB of x; the 44,541-node beam's levels read at most 881 positions back
constexpr int kAhead = 9;    // a node of the beams has at most 9 lower blocks
constexpr int kRingThreads = 512;
// A level of more nodes than the ring has slots (one without lower blocks)
// writes a slot in several passes with no barrier between them: the last one
// stands because the same quad writes them all, in order.
static_assert(kRing % (kRingThreads / 4) == 0, "a ring slot belongs to one quad of the workgroup");
struct SweepLevel {
  int t0, count, base, blocks;
};
struct SweepItem {
  int t, cnt, node;
  bool on;
  double rhs, d[3], v[kAhead][3];
  int sl[kAhead];
};
__global__ void __launch_bounds__(kRingThreads) ica_sweep_ring(const double *__restrict__ lo_val,
                                                               const int *__restrict__ lo_ring,
                                                               const int *__restrict__ lo_cnt,
                                                               const double *__restrict__ dinv,
                                                               const double *__restrict__ rhs,
                                                               const int *__restrict__ node, double *x,
                                                               const SweepLevel *__restrict__ lvl, int n_levels) {
  extern __shared__ double ring[];
  const int kNodes = (int)blockDim.x / 4;
  const int q0 = (int)threadIdx.x / 4, c = min((int)threadIdx.x % 4, 2);
  // Every lane issues every load (past the level's nodes or a node's blocks:
  // its last ones again): with loads under a branch the number in flight is
  // not known where their values are used, and the wait there would be for
  // the next item's loads too.
  auto load = [&](SweepItem &it, const SweepLevel &L, int pass) {
    const int q = min(pass * kNodes + q0, L.count - 1);
    it.on = pass * kNodes + q0 < L.count;
    it.t = L.t0 + q;
    it.cnt = lo_cnt[it.t];
    it.node = node[it.t];
    it.rhs = rhs[3 * (size_t)it.t + c];
#pragma unroll
    for (int e = 0; e < 3; ++e) it.d[e] = dinv[9 * (size_t)it.t + 3 * c + e];
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      it.sl[b] = lo_ring[(size_t)L.base + (size_t)q * L.blocks + b];
      const double *v = lo_val + 9 * ((size_t)L.base + (size_t)max(min(b, L.blocks - 1), 0) * L.count + q) + 3 * c;
#pragma unroll
      for (int e = 0; e < 3; ++e) it.v[b][e] = v[e];
    }
  };
  auto run = [&](const SweepItem &it, const SweepLevel &L, int pass) {
    double r = it.rhs;
    double xb[kAhead][3];
#pragma unroll
    for (int b = 0; b < kAhead; ++b)
#pragma unroll
      for (int e = 0; e < 3; ++e) xb[b][e] = ring[it.sl[b] + e];
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      if (b < it.cnt) {
        r -= it.v[b][0] * xb[b][0];
        r -= it.v[b][1] * xb[b][1];
        r -= it.v[b][2] * xb[b][2];
      }
    }
    for (int b = kAhead; b < it.cnt; ++b) {
      const int q = min(pass * kNodes + q0, L.count - 1);
      const double *xe = ring + lo_ring[(size_t)L.base + (size_t)q * L.blocks + b];
      const double *v = lo_val + 9 * ((size_t)L.base + (size_t)b * L.count + q) + 3 * c;
      r -= v[0] * xe[0];
      r -= v[1] * xe[1];
      r -= v[2] * xe[2];
    }
    const double r0 = quad_lane<0>(r), r1 = quad_lane<1>(r), r2 = quad_lane<2>(r);
    const double xr = it.d[0] * r0 + it.d[1] * r1 + it.d[2] * r2;
    if (it.on) {  // the quad's fourth lane stores the third's value
      ring[3 * (it.t % kRing) + c] = xr;
      x[3 * (size_t)it.node + c] = xr;
    }
  };
  if (n_levels <= 0) return;
  SweepLevel ahead = lvl[min(1, n_levels - 1)];
  // items in order: each level's passes; a barrier ends a level
  auto next = [&](int &lv, int &pass, SweepLevel &L) {  // false past the end
    if ((pass + 1) * kNodes < L.count) {
      ++pass;
      return true;
    }
    if (lv + 1 >= n_levels) return false;
    pass = 0;
    ++lv;
    L = ahead;
    ahead = lvl[min(lv + 1, n_levels - 1)];  // in time for the next level
    return true;
  };
  auto end_level = [&]() {
    // the level's LDS writes before the next level's reads; loads and stores
    // of global memory stay in flight (each x is read back from the LDS)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  SweepItem a, b;
  int la = 0, pa = 0;
  SweepLevel La = lvl[0];
  load(a, La, 0);
  for (;;) {
    int lb = la, pb = pa;
    SweepLevel Lb = La;
    const bool more_b = next(lb, pb, Lb);
    load(b, Lb, pb);  // past the end: the last item again, not run
    run(a, La, pa);
    if (!more_b) break;
    if (lb != la) end_level();
    la = lb;
    pa = pb;
    La = Lb;
    const bool more_a = next(la, pa, La);
    load(a, La, pa);
    run(b, Lb, pb);
    if (!more_a) break;
    if (la != lb) end_level();
  }
}

// The padded blocks' values in the ring sweep's order, gathered once per call
// from their SELL slots (slot < 0: padding, not read).
__global__ void __launch_bounds__(256) ica_ring_vals(const double *__restrict__ val, const int *__restrict__ lo_slot,
                                                     int n_pad, double *__restrict__ lo_val) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_pad) return;
  const long long slot = lo_slot[p];
  if (slot < 0) return;
  const double *v = val + (9 * slot - 8 * (slot % kSlice));
#pragma unroll
  for (int k = 0; k < 9; ++k) lo_val[9 * (size_t)p + k] = v[k * kSlice];
}

// Da^-1 in the sweep's order.
__global__ void __launch_bounds__(256) ica_order_dinv(const double *__restrict__ dinv, const int *__restrict__ node,
                                                      int n_nodes, double *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= 9 * n_nodes) return;
  out[k] = dinv[9 * (size_t)node[k / 9] + k % 9];
}

// ---------------------------------------------------------------- host side

// B = J Da^-1 J^T (CSR, sorted columns) from J over the user's DoFs and the
// inverse blocks in user node order.  Entry (i, k) adds, over the nodes the
// two rows share in ascending order, J_k(v) . (Dinv_v J_i(v)), each product
// left to right.
struct HostCsr {
  std::vector<int> ptr, idx;
  std::vector<double> val;
};

// A row of J as (node, 3-vector) pairs, nodes ascending.
struct RowNodes {
  std::vector<int> node;
  std::vector<double> v;  // 3 per node
};

std::vector<RowNodes> rows_by_node(int m, const int *j_ptr, const int *j_col, const double *j_val) {
  std::vector<RowNodes> rows(m);
  std::vector<std::pair<int, double>> e;
  for (int i = 0; i < m; ++i) {
    e.clear();
    for (int k = j_ptr[i]; k < j_ptr[i + 1]; ++k) e.emplace_back(j_col[k], j_val[k]);
    std::stable_sort(e.begin(), e.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
    RowNodes &R = rows[i];
    for (const auto &pr : e) {
      const int v = pr.first / 3;
      if (R.node.empty() || R.node.back() != v) {
        R.node.push_back(v);
        R.v.insert(R.v.end(), {0.0, 0.0, 0.0});
      }
      R.v[R.v.size() - 3 + pr.first % 3] += pr.second;
    }
  }
  return rows;
}

HostCsr build_b(const std::vector<RowNodes> &rows, int n_nodes, const std::vector<double> &dinv_user) {
  const int m = (int)rows.size();
  // the rows touching each node, ascending, with their slot in that row
  std::vector<std::vector<std::pair<int, int>>> at(n_nodes);
  for (int i = 0; i < m; ++i)
    for (int q = 0; q < (int)rows[i].node.size(); ++q) at[rows[i].node[q]].emplace_back(i, q);
  HostCsr B;
  B.ptr.assign(m + 1, 0);
  std::vector<double> acc(m, 0.0);
  std::vector<char> seen(m, 0);
  std::vector<int> cols;
  for (int i = 0; i < m; ++i) {
    cols.clear();
    const RowNodes &Ri = rows[i];
    for (int q = 0; q < (int)Ri.node.size(); ++q) {
      const int v = Ri.node[q];
      const double *a = &Ri.v[3 * q];
      const double *D = &dinv_user[9 * (size_t)v];
      double w[3];
      for (int r = 0; r < 3; ++r) w[r] = D[3 * r] * a[0] + D[3 * r + 1] * a[1] + D[3 * r + 2] * a[2];
      for (const auto &kq : at[v]) {
        const double *jk = &rows[kq.first].v[3 * kq.second];
        const double d = jk[0] * w[0] + jk[1] * w[1] + jk[2] * w[2];
        if (!seen[kq.first]) {
          seen[kq.first] = 1;
          cols.push_back(kq.first);
          acc[kq.first] = d;
        } else {
          acc[kq.first] += d;
        }
      }
    }
    std::sort(cols.begin(), cols.end());
    for (int k : cols) {
      B.idx.push_back(k);
      B.val.push_back(acc[k]);
      seen[k] = 0;
    }
    B.ptr[i + 1] = (int)B.idx.size();
  }
  return B;
}

// GaussSeidel<true>::solve (ICASolver.h:68-111) on B from lam: rhs = c - Ub lam
// (old lam), then row by row rhs_r -= sum_{k<r} B_rk lam_k (new lam),
// lam_r = max(0, rhs_r / B_rr); stop when |lam - lam_prev| <= tol.  Returns
// the sweeps run.
int pgs(const HostCsr &B, const std::vector<double> &invd, const std::vector<double> &c, std::vector<double> &lam,
        int max_it, double tol, std::vector<double> &rhs, std::vector<double> &pre) {
  const int m = (int)c.size();
  for (int it = 0; it < max_it; ++it) {
    pre = lam;
    for (int r = 0; r < m; ++r) {
      double u = 0.0;
      for (int k = B.ptr[r]; k < B.ptr[r + 1]; ++k)
        if (B.idx[k] > r) u += B.val[k] * lam[B.idx[k]];
      rhs[r] = c[r] - u;
    }
    for (int r = 0; r < m; ++r) {
      for (int k = B.ptr[r]; k < B.ptr[r + 1]; ++k)
        if (B.idx[k] < r) rhs[r] -= lam[B.idx[k]] * B.val[k];
      const double v = rhs[r] * invd[r];
      lam[r] = v > 0 ? v : 0;
    }
    double s = 0.0;
    for (int r = 0; r < m; ++r) s += (lam[r] - pre[r]) * (lam[r] - pre[r]);
    if (std::sqrt(s) <= tol) return it + 1;
  }
  return max_it;
}

}  // namespace
}  // namespace mprgp

using namespace mprgp;

extern "C" int mprgp_ica_solve(mprgp_qp *q, int m, const int *j_ptr, const int *j_col, const double *j_val,
                               const double *p, double tol, int max_it, int gs_max_it, double gs_tol,
                               double *lambda, int *pgs_sweeps, mprgp_stats *stats) {
  MPRGP_TRY
  if (!q || m < 0 || (m > 0 && (!j_ptr || !j_col || !j_val || !p))) return fail(MPRGP_EBADINPUT, "bad ICA arguments");
  if (!(tol == tol) || max_it < 0 || gs_max_it < 0 || !(gs_tol == gs_tol))
    return fail(MPRGP_EBADINPUT, "bad ICA tolerances or iteration limits");
  if (!q->has_rhs || !q->has_x) return fail(MPRGP_ESTATE, "rhs and x must be set");
  MPRGP_NOT_BUSY(q);
  mprgp_ctx *ctx = q->ctx;
  const mprgp_matrix *A = q->A;
  MPRGP_HIP(hipSetDevice(ctx->device));
  std::lock_guard<std::recursive_mutex> lk_(ctx->mu);
  const int nn = q->n, n = 3 * nn;
  RowsInternal Ri;
  if (int rc = rows_to_internal(A, m, j_ptr, j_col, j_val, p, Ri)) return rc;
  const int nnz = m > 0 ? j_ptr[m] : 0;
  hipStream_t s = ctx->stream;

  // dependency levels of the sweep from the matrix structure (user order)
  std::vector<int> col((size_t)A->slots);
  MPRGP_HIP(hipMemcpyAsync(col.data(), A->d_col, sizeof(int) * col.size(), hipMemcpyDeviceToHost, s));
  MPRGP_HIP(hipStreamSynchronize(s));
  std::vector<int> level(nn, 0);
  int n_levels = nn > 0 ? 1 : 0;
  for (int u = 0; u < nn; ++u) {
    const int i = A->iperm[u], sl = i / kSlice, l = i % kSlice;
    const int b0 = A->sl_off_h[sl], W = (A->sl_off_h[sl + 1] - b0) / kSlice;
    int lv = 0;
    for (int k = 0; k < W; ++k) {
      const int c = col[(size_t)b0 + (size_t)k * kSlice + l];
      const int uc = A->perm[c];
      if (uc < u) lv = std::max(lv, level[uc] + 1);
    }
    level[u] = lv;
    n_levels = std::max(n_levels, lv + 1);
  }
  std::vector<int> lvl_ptr(n_levels + 1, 0), lvl_node(nn);
  for (int u = 0; u < nn; ++u) lvl_ptr[level[u] + 1]++;
  for (int lv = 0; lv < n_levels; ++lv) lvl_ptr[lv + 1] += lvl_ptr[lv];
  {
    std::vector<int> fill(lvl_ptr.begin(), lvl_ptr.end() - 1);
    for (int u = 0; u < nn; ++u) lvl_node[fill[level[u]]++] = A->iperm[u];
  }
  // each level-ordered node's lower blocks (nodes before it), in block
  // order: SELL slot and column
  std::vector<int> lo_ptr(nn + 1, 0), lo_slot, lo_col, pos(nn);
  for (int t = 0; t < nn; ++t) pos[lvl_node[t]] = t;
  for (int t = 0; t < nn; ++t) {
    const int i = lvl_node[t], u = A->perm[i], sl = i / kSlice, l = i % kSlice;
    const int b0 = A->sl_off_h[sl], W = (A->sl_off_h[sl + 1] - b0) / kSlice;
    for (int k = 0; k < W; ++k) {
      const int slot = b0 + k * kSlice + l, c = col[(size_t)slot];
      if (A->perm[c] < u) {
        lo_slot.push_back(slot);
        lo_col.push_back(c);
      }
    }
    lo_ptr[t + 1] = (int)lo_slot.size();
  }
  const size_t n_lo = lo_slot.size();
  // the ring sweep's levels, if every column a level reads is within kRing
  // positions of the level's end and the padded blocks stay few
  std::vector<SweepLevel> lvl(n_levels);
  std::vector<int> lo_cnt(nn), ring_slot, lo_ring;  // the padded blocks' SELL slots and ring slots
  bool use_ring = true;
  int ring_threads = 64;
  size_t n_pad = 0;
  for (int lv = 0; lv < n_levels; ++lv) {
    int most = 0;
    for (int t = lvl_ptr[lv]; t < lvl_ptr[lv + 1]; ++t) {
      lo_cnt[t] = lo_ptr[t + 1] - lo_ptr[t];
      most = std::max(most, lo_cnt[t]);
      for (int e = lo_ptr[t]; e < lo_ptr[t + 1]; ++e)
        use_ring = use_ring && lvl_ptr[lv + 1] - 1 - pos[lo_col[e]] < kRing;
    }
    lvl[lv] = SweepLevel{lvl_ptr[lv], lvl_ptr[lv + 1] - lvl_ptr[lv], (int)n_pad, most};
    n_pad += (size_t)most * lvl[lv].count;
    use_ring = use_ring && 9 * n_pad < 0x7fffffff;
  }
  use_ring = use_ring && n_pad <= 3 * n_lo + 1024;
  if (use_ring) {
    // a level without lower blocks reads one block column past its base, a
    // node's kAhead slots may run past its own
    int widest = 0;
    for (const SweepLevel &L : lvl) widest = std::max(widest, L.count);
    n_pad += widest + kAhead;
    ring_threads = std::min(kRingThreads, (4 * widest + 63) / 64 * 64);
    ring_slot.assign(n_pad, -1);
    lo_ring.assign(n_pad, 0);
    for (const SweepLevel &L : lvl)
      for (int qn = 0; qn < L.count; ++qn)
        for (int b = 0; b < lo_cnt[L.t0 + qn]; ++b) {
          const size_t e = lo_ptr[L.t0 + qn] + b;
          ring_slot[(size_t)L.base + (size_t)b * L.count + qn] = lo_slot[e];
          lo_ring[(size_t)L.base + (size_t)qn * L.blocks + b] = 3 * (pos[lo_col[e]] % kRing);
        }
  }

  // device block: Da^-1, levels, the lower blocks and their values, J and
  // J^T, J u, lambda, dot partials.  The ring sweep's, with up to three times
  // the blocks and a second Da^-1, is the larger; where it is refused, the
  // sweep that reads x from memory takes its place.
  const size_t parts = ((size_t)n + 255) / 256 + 1;
  const size_t common = sizeof(double) * (2 * (size_t)nnz + 2 * (size_t)m + parts + 8) +
                        sizeof(int) * ((size_t)m + 1 + 2 * (size_t)nnz + (size_t)n + 1) + 1024;
  size_t bytes = common + sizeof(double) * (18 * (size_t)nn + 9 * n_pad) +
                 sizeof(int) * (3 * (size_t)nn + 1 + 2 * n_pad) + sizeof(SweepLevel) * (size_t)n_levels;
  void *blk = nullptr;
  use_ring = use_ring && ctx->alloc(&blk, bytes) == MPRGP_OK;
  if (!use_ring) {
    bytes = common + sizeof(double) * (9 * (size_t)nn + 9 * n_lo) +
            sizeof(int) * ((size_t)n_levels + 1 + 2 * (size_t)nn + 1 + 2 * n_lo);
    if (int rc = ctx->alloc(&blk, bytes)) return rc;
  }
  // the blocks as the chosen sweep reads them
  const size_t n_blk = use_ring ? n_pad : n_lo;
  const std::vector<int> &blk_slot = use_ring ? ring_slot : lo_slot, &blk_col = use_ring ? lo_ring : lo_col;
  struct Release {  // on every exit: the stream's work on the block ends first
    mprgp_ctx *c;
    void *p;
    size_t b;
    ~Release() {
      (void)hipStreamSynchronize(c->stream);
      c->release(p, b);
    }
  } release_{ctx, blk, bytes};
  char *b8 = (char *)blk;
  auto carve = [&](size_t sz) {
    uintptr_t u = ((uintptr_t)b8 + 7) & ~(uintptr_t)7;
    b8 = (char *)(u + sz);
    return (void *)u;
  };
  double *d_dinv = (double *)carve(sizeof(double) * 9 * (size_t)nn);
  double *d_jv = (double *)carve(sizeof(double) * nnz);
  double *d_tv = (double *)carve(sizeof(double) * nnz);
  double *d_jx = (double *)carve(sizeof(double) * (m + 1));
  double *d_lam = (double *)carve(sizeof(double) * (m + 1));
  double *d_part = (double *)carve(sizeof(double) * parts);
  int *d_lvl_ptr = use_ring ? nullptr : (int *)carve(sizeof(int) * (n_levels + 1));
  int *d_lvl_node = (int *)carve(sizeof(int) * (size_t)nn);
  double *d_lo_val = (double *)carve(sizeof(double) * 9 * n_blk);
  int *d_lo_ptr = (int *)carve(sizeof(int) * ((size_t)nn + 1));
  int *d_lo_slot = (int *)carve(sizeof(int) * n_blk);
  int *d_lo_col = (int *)carve(sizeof(int) * n_blk);
  double *d_dinv_t = use_ring ? (double *)carve(sizeof(double) * 9 * (size_t)nn) : nullptr;
  SweepLevel *d_lvl = use_ring ? (SweepLevel *)carve(sizeof(SweepLevel) * (size_t)n_levels) : nullptr;
  int *d_pos = use_ring ? (int *)carve(sizeof(int) * (size_t)nn) : nullptr;
  int *d_jp = (int *)carve(sizeof(int) * (m + 1));
  int *d_jc = (int *)carve(sizeof(int) * nnz);
  int *d_tp = (int *)carve(sizeof(int) * (n + 1));
  int *d_tc = (int *)carve(sizeof(int) * nnz);
  if (m > 0) {
    MPRGP_HIP(hipMemcpyAsync(d_jp, j_ptr, sizeof(int) * (m + 1), hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_jc, Ri.jc.data(), sizeof(int) * nnz, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_jv, j_val, sizeof(double) * nnz, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_tc, Ri.tc.data(), sizeof(int) * nnz, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_tv, Ri.tv.data(), sizeof(double) * nnz, hipMemcpyHostToDevice, s));
  }
  MPRGP_HIP(hipMemcpyAsync(d_tp, Ri.tptr.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, s));
  MPRGP_HIP(hipMemcpyAsync(d_lvl_node, lvl_node.data(), sizeof(int) * (size_t)nn, hipMemcpyHostToDevice, s));
  if (use_ring) {
    MPRGP_HIP(hipMemcpyAsync(d_lo_ptr, lo_cnt.data(), sizeof(int) * (size_t)nn, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_lvl, lvl.data(), sizeof(SweepLevel) * (size_t)n_levels, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_pos, pos.data(), sizeof(int) * (size_t)nn, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipFuncSetAttribute((const void *)ica_sweep_ring, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  3 * kRing * (int)sizeof(double)));
  } else {
    MPRGP_HIP(hipMemcpyAsync(d_lvl_ptr, lvl_ptr.data(), sizeof(int) * (n_levels + 1), hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_lo_ptr, lo_ptr.data(), sizeof(int) * ((size_t)nn + 1), hipMemcpyHostToDevice, s));
  }
  if (n_blk > 0) {
    MPRGP_HIP(hipMemcpyAsync(d_lo_slot, blk_slot.data(), sizeof(int) * n_blk, hipMemcpyHostToDevice, s));
    MPRGP_HIP(hipMemcpyAsync(d_lo_col, blk_col.data(), sizeof(int) * n_blk, hipMemcpyHostToDevice, s));
  }
  const int blocks = (nn + 255) / 256;
  if (nn > 0) {
    ica_dinv<<<blocks, 256, 0, s>>>(A->d_sl_off, A->d_col, A->d_val, nn, d_dinv);
    MPRGP_HIP(hipGetLastError());
  }
  if (use_ring && nn > 0) {
    ica_order_dinv<<<(9 * nn + 255) / 256, 256, 0, s>>>(d_dinv, d_lvl_node, nn, d_dinv_t);
    MPRGP_HIP(hipGetLastError());
  }
  if (n_blk > 0) {
    const unsigned grid = (unsigned)((n_blk + 255) / 256);
    if (use_ring) ica_ring_vals<<<grid, 256, 0, s>>>(A->d_val, d_lo_slot, (int)n_blk, d_lo_val);
    else ica_lower_vals<<<grid, 256, 0, s>>>(A->d_val, d_lo_slot, (int)n_blk, d_lo_val);
    MPRGP_HIP(hipGetLastError());
  }
  // B = J Da^-1 J^T on the host, from the inverse blocks in user order
  std::vector<RowNodes> rows;
  HostCsr B;
  std::vector<double> invd(m, 0.0), c(m), lam(m, 0.0), rhs(m), pre(m);
  if (m > 0) {
    std::vector<double> dinv((size_t)9 * nn), dinv_user((size_t)9 * nn);
    MPRGP_HIP(hipMemcpyAsync(dinv.data(), d_dinv, sizeof(double) * dinv.size(), hipMemcpyDeviceToHost, s));
    MPRGP_HIP(hipStreamSynchronize(s));
    for (int u = 0; u < nn; ++u)
      std::copy(&dinv[9 * (size_t)A->iperm[u]], &dinv[9 * (size_t)A->iperm[u]] + 9, &dinv_user[9 * (size_t)u]);
    rows = rows_by_node(m, j_ptr, j_col, j_val);
    B = build_b(rows, nn, dinv_user);
    for (int r = 0; r < m; ++r)
      for (int k = B.ptr[r]; k < B.ptr[r + 1]; ++k)
        if (B.idx[k] == r) invd[r] = 1.0 / B.val[k];
  }
  double *u = q->z, *jtl = q->phi, *rh = q->beta, *e = q->ap;
  const double *x_c = q->x;
  // J u and the residual as read back (d_jx, m + 1 doubles), lambda: pinned
  // where that is to be had.  Every iteration waits for the readback before
  // lambda is written again.
  struct Pinned {
    double *p = nullptr;
    ~Pinned() {
      if (p) (void)hipHostFree(p);
    }
  } pin;
  std::vector<double> pageable;
  if (hipHostMalloc((void **)&pin.p, sizeof(double) * (2 * (size_t)m + 1), hipHostMallocDefault) != hipSuccess) {
    pin.p = nullptr;
    (void)hipGetLastError();
    pageable.resize(2 * (size_t)m + 1);
  }
  double *h_jx = pin.p ? pin.p : pageable.data(), *h_lam = h_jx + m + 1, *d_r2 = d_jx + m;
  Release drain_{ctx, nullptr, 0};  // before that memory goes: an upload from it may be queued
  MPRGP_HIP(hipMemsetAsync(jtl, 0, sizeof(double) * n, s));
  MPRGP_HIP(hipMemsetAsync(d_jx, 0, sizeof(double) * ((size_t)m + 1), s));
  MPRGP_HIP(hipEventRecord(ctx->t0, s));
  int it = 0, sweeps = 0;
  bool met = false;
  double residual = -1.0;
  // J u for the next c = p + J Da^-1 (LaUa x - b), queued behind the sweep
  // that makes its x, so that one wait per iteration brings it back with the
  // residual (after the last sweep it is not used)
  auto queue_ju = [&]() -> int {
    ica_rows<<<blocks, 256, 0, s>>>(A->d_sl_off, A->d_col, A->d_val, A->d_perm, x_c, q->b, jtl, d_dinv, u, nn,
                                    kOffDiag, nullptr);
    MPRGP_HIP(hipGetLastError());
    MPRGP_HIP(launch_csr_mul(s, m, d_jp, d_jc, d_jv, u, d_jx));
    return MPRGP_OK;
  };
  auto read_back = [&]() -> int {
    MPRGP_HIP(hipMemcpyAsync(h_jx, d_jx, sizeof(double) * ((size_t)m + 1), hipMemcpyDeviceToHost, s));
    MPRGP_HIP(hipStreamSynchronize(s));
    return MPRGP_OK;
  };
  if (m > 0 && max_it > 0) {
    if (int rc = queue_ju()) return rc;
    if (int rc = read_back()) return rc;
  }
  for (it = 0; it < max_it; ++it) {
    if (m > 0) {
      for (int i = 0; i < m; ++i) c[i] = p[i] + h_jx[i];
      sweeps += pgs(B, invd, c, lam, gs_max_it, gs_tol, rhs, pre);
      std::copy(lam.begin(), lam.end(), h_lam);
      MPRGP_HIP(hipMemcpyAsync(d_lam, h_lam, sizeof(double) * m, hipMemcpyHostToDevice, s));
      MPRGP_HIP(launch_csr_mul(s, n, d_tp, d_tc, d_tv, d_lam, jtl));
    }
    if (nn > 0) {
      ica_rows<<<blocks, 256, 0, s>>>(A->d_sl_off, A->d_col, A->d_val, A->d_perm, x_c, q->b, jtl, d_dinv, rh, nn,
                                      kUpper, use_ring ? d_pos : nullptr);
      MPRGP_HIP(hipGetLastError());
      if (use_ring)
        ica_sweep_ring<<<1, ring_threads, 3 * kRing * sizeof(double), s>>>(d_lo_val, d_lo_col, d_lo_ptr, d_dinv_t, rh,
                                                                           d_lvl_node, q->x, d_lvl, n_levels);
      else
        ica_sweep<<<1, kSweepThreads, 0, s>>>(d_lo_val, d_lo_col, d_lo_ptr, d_dinv, rh, q->x, d_lvl_ptr,
                                              d_lvl_node, n_levels);
      MPRGP_HIP(hipGetLastError());
      ica_rows<<<blocks, 256, 0, s>>>(A->d_sl_off, A->d_col, A->d_val, A->d_perm, x_c, q->b, jtl, d_dinv, e, nn,
                                      kResidual, nullptr);
      MPRGP_HIP(hipGetLastError());
    }
    MPRGP_HIP(launch_dot(s, e, e, (size_t)n, d_part, d_r2));
    if (m > 0 && it + 1 < max_it)
      if (int rc = queue_ju()) return rc;
    if (int rc = read_back()) return rc;
    residual = std::sqrt(h_jx[m]);
    if (residual <= tol) {
      met = true;
      break;
    }
  }
  MPRGP_HIP(hipEventRecord(ctx->t1, s));
  MPRGP_HIP(hipStreamSynchronize(s));
  float ms = 0.f;
  MPRGP_HIP(hipEventElapsedTime(&ms, ctx->t0, ctx->t1));
  if (lambda)
    for (int i = 0; i < m; ++i) lambda[i] = lam[i];
  if (pgs_sweeps) *pgs_sweeps = sweeps;
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    stats->code = met ? 0 : -1;
    stats->iterations = it;
    stats->residual = residual;
    stats->elapsed_ms = ms;
    stats->error_bound = -1.0;
  }
  if (!std::isfinite(residual) && max_it > 0) return fail(MPRGP_ENAN, "ICA residual is not finite");
  return met ? MPRGP_OK : MPRGP_NOT_CONVERGED;
  MPRGP_CATCH
}
