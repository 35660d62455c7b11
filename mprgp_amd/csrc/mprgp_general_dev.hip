// mprgp_general_dev.hip -- the main loop of the coupled-row solve
// (MPRGPMonotonic::solve with GeneralConProjector, MPRGPSolver.h:412-454,
// MPRGPProjection.h:400-520) in one workgroup, for systems of at most
// kGenMaxNodes nodes whose rows form components of at most kGenBlock rows,
// where one CU is the faster way (mprgp_general.h).
//
// Driven from the host, an iteration is about 50 launches of small kernels and
// five waits, nearly all of its time.  Here the vectors stay where they are
// (the QP's buffers), the phases of an iteration are separated by workgroup
// barriers, and the projection's small QPs and the active rows' factors are
// computed by one wavefront per component.  A solve of 1,001 iterations on a
// 525-node beam with 537 rows: 370 ms from the host, 112 ms here (an expansion
// step 295,000 cycles: five products with A at 19,000-21,000, three
// projections at 26,000-34,000); 1,476 nodes 547 and 228 ms; 2,499 nodes 570
// and 271 ms.  The products are bound by the CU's load path, which takes
// about 32 bytes of the matrix a cycle, so their share grows with the size.
//
// Every value is formed as the host-driven loop forms it: products with J and
// A by fused multiply-adds in stored order, the dot products as one sum tree
// per 256 entries and a tree over those, the components' QPs and factors
// without fused operations, so that both loops give the same bits.
#include <hip/hip_runtime.h>

#include "mprgp_general.h"

#pragma clang fp contract(off)

namespace mprgp {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kSlice;
constexpr int K = kGenBlock;
constexpr int kUnroll = 3;  // blocks of a row in flight; 4 do not fit the registers of 16 wavefronts

// The arguments lie in device memory and are read with scalar loads, by each
// of the functions below what it needs: as one body, all phases in line, the
// kernel is 11,000 instructions, more than the instruction cache holds.
using Args = const __attribute__((address_space(4))) GenArgs;

struct Block {
  double vec[3 * kGenMaxNodes];  // the vector a product gathers from
  double red[2][kWaves];
  double sum[5];
  int infeasible, fail, spec;
};
using Shared = __attribute__((address_space(3))) Block;

template <class T>
__device__ __forceinline__ T *uniform(T *p) {  // p, the same in all lanes, in scalar registers
  const auto u = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return (T *)((unsigned long long)hi << 32 | lo);
}
template <class T>
using Mem = __attribute__((address_space(1))) T *;
template <class T>
__device__ __forceinline__ Mem<T> mem(T *p) {  // p is device memory
  return (Mem<T>)p;
}

// A component's QP is solved by one wavefront, all lanes alike: the block of
// J J^T is one load, entry e in lane e, read from there, and the branches on
// the free rows are scalar.  (One lane per component, entries loaded where the
// branches need them, made the solve 128 ms instead of 110.)
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Place of entry (i, j), j <= i, of a packed lower triangle.
__host__ __device__ constexpr int tri(int i, int j) { return i * (i + 1) / 2 + j; }
constexpr int kTri = K * (K + 1) / 2;

// Cholesky of the rows `on` of the block G (lower factor, packed) and the
// forward substitution y = L^-1 b, without the rows that are off; false if a
// pivot is not positive.  Rows below `from` are as an earlier call left them:
// a row of the factor depends on the rows above it alone.
__device__ __forceinline__ bool factor(double G, unsigned on, int from, const double (&b)[K], double (&L)[kTri],
                                       double (&y)[K]) {
#pragma unroll
  for (int i = 0; i < K; ++i)
    if (i >= from && (on >> i & 1)) {
      double d = lane_value(G, i * K + i), t = b[i];
#pragma unroll
      for (int j = 0; j < i; ++j)
        if (on >> j & 1) {
          double v = lane_value(G, i * K + j);
#pragma unroll
          for (int p = 0; p < j; ++p)
            if (on >> p & 1) v -= L[tri(i, p)] * L[tri(j, p)];
          v = v / L[tri(j, j)];
          L[tri(i, j)] = v;
          d -= v * v;
          t -= v * y[j];
        }
      if (!(d > 0.0)) return false;
      d = sqrt(d);
      L[tri(i, i)] = d;
      y[i] = t / d;
    }
  return true;
}
// s = L^-T y over the rows `on`
__device__ __forceinline__ void back(const double (&L)[kTri], unsigned on, const double (&y)[K], double (&s)[K]) {
#pragma unroll
  for (int i = K - 1; i >= 0; --i) {
    s[i] = 0.0;
    if (on >> i & 1) {
      double v = y[i];
#pragma unroll
      for (int p = i + 1; p < K; ++p)
        if (on >> p & 1) v -= L[tri(p, i)] * s[p];
      s[i] = v / L[tri(i, i)];
    }
  }
}
// out[row_i] = v[i], lane i storing it
__device__ __forceinline__ void put_rows(int r, const double (&v)[K], Mem<double> out) {
  const int lane = threadIdx.x % kSlice;
  double mine = 0.0;
#pragma unroll
  for (int i = 0; i < K; ++i)
    if (lane == i) mine = v[i];
  if (lane < K && r >= 0) out[r] = mine;
}

// One component (its rows, -1: none): out = argmin 1/2 l'Gl - h'l, l >= 0,
// with h = c - jv over all rows (a projection) or h = jv over the face's rows
// (BETA); the rows left out get 0.  Primal active set on the free
// rows, as the host-driven loop's qp_nonneg; false if a free block is not
// positive definite.
__device__ __forceinline__ bool component_qp(Mem<const double> g, Mem<const int> row, Mem<const double> jv,
                                             Mem<const double> c, bool all, Mem<const unsigned char> face, double tol,
                                             Mem<double> out) {
  const int lane = threadIdx.x % kSlice;
  const double G = g[min(lane, K * K - 1)];
  const int r = lane < K ? row[min(lane, K - 1)] : -1;
  const int at = max(r, 0);
  const double v = jv[at];
  const bool in = r >= 0 && (all || face[at]);
  const double hl = all ? c[at] - v : v;
  const unsigned allowed = (unsigned)__ballot(in);
  double h[K], lam[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    h[i] = lane_value(hl, i);
    lam[i] = 0.0;
  }
  const int k = __popc(allowed);
  unsigned free_ = 0;
  int from = K;  // the lowest row whose place in the free set changed since the factor was formed
  double L[kTri], y[K], s[K];
  bool ok = k == 0;
  for (int outer = 0; outer < 10 * k + 10 && !ok; ++outer) {
    int best = -1;
    double wbest = tol;
#pragma unroll
    for (int i = 0; i < K; ++i)
      if (allowed >> i & 1) {
        double w = h[i];
#pragma unroll
        for (int j = 0; j < K; ++j)
          if (allowed >> j & 1) w -= lane_value(G, i * K + j) * lam[j];
        if (!(free_ >> i & 1) && w > wbest) {
          wbest = w;
          best = i;
        }
      }
    best = __builtin_amdgcn_readfirstlane(best);
    if (best < 0) {
      ok = true;
      break;
    }
    free_ |= 1u << best;
    from = min(from, best);
    bool bad = false;
    for (int inner = 0; inner <= k; ++inner) {
      if (!factor(G, free_, from, h, L, y)) {
        bad = true;
        break;
      }
      from = K;
      back(L, free_, y, s);
      double step = 1.0;
      int hit = -1;
#pragma unroll
      for (int i = 0; i < K; ++i)
        if ((free_ >> i & 1) && s[i] <= 0.0) {
          const double t = lam[i] / (lam[i] - s[i]);
          if (t < step) {
            step = t;
            hit = i;
          }
        }
      hit = __builtin_amdgcn_readfirstlane(hit);
      if (hit < 0) {
#pragma unroll
        for (int i = 0; i < K; ++i) lam[i] = s[i];
        break;
      }
      unsigned left = free_;
#pragma unroll
      for (int i = 0; i < K; ++i)
        if (free_ >> i & 1) {
          lam[i] += step * (s[i] - lam[i]);
          if (i == hit || lam[i] <= 0.0) {
            left &= ~(1u << i);
            lam[i] = 0.0;
          }
        }
      left = __builtin_amdgcn_readfirstlane(left);
      from = __ffs(free_ ^ left) - 1;
      free_ = left;
    }
    if (bad) break;
  }
  put_rows(r, lam, out);
  return ok;
}

// PHI's multipliers of one component from J g: (J_a J_a^T) l = -J_a g over
// the face's rows.
__device__ __forceinline__ bool component_phi(Mem<const double> g, Mem<const int> row, Mem<const double> jg,
                                              Mem<const unsigned char> face, Mem<double> out) {
  const int lane = threadIdx.x % kSlice;
  const double G = g[min(lane, K * K - 1)];
  const int r = lane < K ? row[min(lane, K - 1)] : -1;
  const int at = max(r, 0);
  const bool in = r >= 0 && face[at];
  const double ll = in ? -jg[at] : 0.0;
  const unsigned on = (unsigned)__ballot(in);
  double b[K], l[K], y[K], L[kTri];
#pragma unroll
  for (int i = 0; i < K; ++i) b[i] = lane_value(ll, i);
  const bool ok = factor(G, on, 0, b, L, y);
  if (ok) back(L, on, y, l);
  else
    for (int i = 0; i < K; ++i) l[i] = 0.0;
  put_rows(r, l, out);
  return ok;
}

// Sum of v over the wavefront's lanes as a tree of halves (lane 0).
__device__ __forceinline__ double halves(double v) {
#pragma unroll
  for (int w = kSlice / 2; w > 0; w >>= 1) v += __shfl_down(v, w, kSlice);
  return v;
}

// Row i of a CSR matrix times v, four entries loaded at a time.
__device__ __forceinline__ double csr_row(Mem<const int> ptr, Mem<const int> col, Mem<const double> val,
                                          Mem<const double> v, int i) {
  const int b = ptr[i], e = ptr[i + 1];
  double s = 0.0;
  for (int k = b; k < e; k += 4) {
    double w[4], q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = min(k + u, e - 1);
      w[u] = val[at];
      q[u] = v[col[at]];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + u < e) s = __builtin_fma(w[u], q[u], s);
  }
  return s;
}
// (J v)_i and (J^T lam)_i
__device__ __forceinline__ double j_row(Args *a, const double *v, int i) {
  return csr_row(mem(a->jp), mem(a->jc), mem(a->jv), mem(v), i);
}
__device__ __forceinline__ double jt_row(Args *a, const double *lam, int i) {
  return csr_row(mem(a->tp), mem(a->tc), mem(a->tv), mem(lam), i);
}

// o0 = J v0, o1 = J v1
__device__ __noinline__ void j_mul(Args *a_, const double *v0, double *o0, const double *v1, double *o1) {
  Args *a = uniform(a_);
  const int m = a->m;
  for (int i = threadIdx.x; i < m; i += kThreads) {
    mem(o0)[i] = j_row(a, v0, i);
    if (o1) mem(o1)[i] = j_row(a, v1, i);
  }
}

// out = A v and, where asked for, g = A v - b; one wavefront per slice.  v
// is copied to LDS first: gathered from memory, a node's 24 bytes cost the
// cache as many cycles as the matrix entries they multiply (525 nodes: 25,000
// cycles a product, from LDS 19,300).  Ends with a barrier.
__device__ __noinline__ void product(Args *a_, Shared *sh, const double *v, double *out_, double *g_) {
  Args *a = uniform(a_);
  const auto b = mem(a->b);
  const auto out = mem(uniform(out_)), g = mem(uniform(g_));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kSlice), lane = threadIdx.x % kSlice;
  const int n_slices = a->n_slices, n_nodes = a->n_nodes, n = a->n;
  for (int i = threadIdx.x; i < n; i += kThreads) sh->vec[i] = mem(v)[i];
  __syncthreads();
  for (int s = wave; s < n_slices; s += kWaves) {
    const int r = s * kSlice + lane;
    const int b0 = mem(a->sl_off)[s], W = (mem(a->sl_off)[s + 1] - b0) / kSlice;
    const auto cp = mem(a->col) + b0 + lane;
    const auto vp = mem(a->val) + (size_t)b0 * 9 + lane;
    double x = 0.0, y = 0.0, z = 0.0;
    int j[kUnroll] = {};
    if (W > 0)
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) j[u] = cp[min(u, W - 1) * kSlice];
    for (int k0 = 0; k0 < W; k0 += kUnroll) {
      double e[kUnroll][9];
      int next[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
#pragma unroll
        for (int i = 0; i < 9; ++i) e[u][i] = vp[(size_t)min(k0 + u, W - 1) * (9 * kSlice) + i * kSlice];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) next[u] = cp[min(k0 + kUnroll + u, W - 1) * kSlice];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
        if (k0 + u < W) {
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const double q = sh->vec[3 * j[u] + i];
            x = __builtin_fma(e[u][i], q, x);
            y = __builtin_fma(e[u][3 + i], q, y);
            z = __builtin_fma(e[u][6 + i], q, z);
          }
        }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) j[u] = next[u];
    }
    if (r < n_nodes) {
      const int o = 3 * r;
      out[o] = x;
      out[o + 1] = y;
      out[o + 2] = z;
      if (g) {
        g[o] = x - b[o];
        g[o + 1] = y - b[o + 1];
        g[o + 2] = z - b[o + 2];
      }
    }
  }
  __syncthreads();
}

// sh->sum[first + j] = sums of f(i, p)'s p[j] over the entries i: a wavefront
// per 256 entries, then a wavefront per sum.
template <int N, class F>
__device__ __forceinline__ void sums(Args *a, Shared *sh, int first, F f) {
  const int wave = threadIdx.x / kSlice, lane = threadIdx.x % kSlice;
  const int n = a->n, chunks = (n + 255) / 256;
  const auto part = mem(a->part);
  for (int c = wave; c < chunks; c += kWaves) {
    double p[4][N];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = c * 256 + u * 64 + lane;
#pragma unroll
      for (int j = 0; j < N; ++j) p[u][j] = 0.0;
      if (i < n) f(i, p[u]);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const double s = halves((p[0][j] + p[2][j]) + (p[1][j] + p[3][j]));
      if (lane == 0) part[j * chunks + c] = s;
    }
  }
  __syncthreads();
  if (wave < N) {
    double q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      q[u] = 0.0;
      for (int i = u * 64 + lane; i < chunks; i += 256) q[u] = q[u] + part[wave * chunks + i];
    }
    const double s = halves((q[0] + q[2]) + (q[1] + q[3]));
    if (lane == 0) sh->sum[first + wave] = s;
  }
  __syncthreads();
}
// u.v and w.t
__device__ __noinline__ void dots(Args *a_, Shared *sh, int first, const double *u, const double *v, const double *w,
                                  const double *t) {
  Args *a = uniform(a_);
  sums<2>(a, sh, first, [&](int i, double *p) {
    p[0] = mem(u)[i] * mem(v)[i];
    p[1] = mem(w)[i] * mem(t)[i];
  });
}

// The components' multipliers.  A projection: lam from h = c - J v (J v in j1)
// over all rows; the loop head: lam from BETA's h = J beta (j1) over the face's
// rows, and lam2 from the projection of t2 (j2), at once.  A wavefront
// per component of several rows, a thread per single row.  The freeing threshold is 1e-14 max |h| of
// the whole QP.  A block that is not positive definite sets fail, or spec for
// t2's projection, which counts only if the proportioning test is evaluated.
__device__ __noinline__ void multipliers(Args *a_, Shared *sh, bool at_head) {
  Args *a = uniform(a_);
  const int m = a->m, tid = threadIdx.x, lane = tid % kSlice;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kSlice);
  const auto c = mem(a->c), jb = mem((const double *)a->j1), jp = at_head ? mem((const double *)a->j2) : jb;
  const auto lb = mem(a->lam), lp = at_head ? mem(a->lam2) : lb;
  const auto face = mem((const unsigned char *)a->face);
  double top[2] = {0.0, 0.0};
  for (int i = tid; i < m; i += kThreads) {
    top[0] = fmax(top[0], fabs(c[i] - jp[i]));
    if (at_head && face[i]) top[1] = fmax(top[1], fabs(jb[i]));
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int w = kSlice / 2; w > 0; w >>= 1) top[q] = fmax(top[q], __shfl_xor(top[q], w, kSlice));
    if (lane == 0) sh->red[q][wave] = top[q];
  }
  __syncthreads();
  double tol[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    double t = sh->red[q][lane % kWaves];
#pragma unroll
    for (int w = kWaves / 2; w > 0; w >>= 1) t = fmax(t, __shfl_xor(t, w, kSlice));
    tol[q] = 1e-14 * (t > 0.0 ? t : 1.0);
  }
  const int n_big = a->n_big, n_one = a->n_one, sets = at_head ? 2 : 1;
  for (int q = wave; q < n_big * sets; q += kWaves) {
    const bool beta = q >= n_big;
    const int k = beta ? q - n_big : q;
    if (!component_qp(mem(a->big_g) + (size_t)k * K * K, mem(a->big_row) + k * K, beta ? jb : jp, c, !beta, face,
                      beta ? tol[1] : tol[0], beta ? lb : lp))
      *(at_head && !beta ? &sh->spec : &sh->fail) = 1;
  }
  for (int k = kThreads - 1 - tid; k < n_one; k += kThreads) {
    const int r = mem(a->one_row)[k];
    const double g = mem(a->one_g)[k], d = sqrt(g);
    const double hp = c[r] - jp[r];
    double l = 0.0;
    if (hp > tol[0]) {
      if (g > 0.0) l = hp / d / d;
      else *(at_head ? &sh->spec : &sh->fail) = 1;
    }
    lp[r] = l;
    if (at_head) {
      l = 0.0;
      if (face[r] && jb[r] > tol[1]) {
        if (g > 0.0) l = jb[r] / d / d;
        else sh->fail = 1;
      }
      lb[r] = l;
    }
  }
  __syncthreads();
}

// lam = PHI's multipliers of J g (in j2): (J_a J_a^T) l = -J_a g
__device__ __noinline__ void phi_multipliers(Args *a_, Shared *sh) {
  Args *a = uniform(a_);
  const int n_big = a->n_big, n_one = a->n_one, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kSlice);
  const auto face = mem((const unsigned char *)a->face);
  const auto jg = mem((const double *)a->j2);
  const auto lam = mem(a->lam);
  bool ok = true;
  for (int k = wave; k < n_big; k += kWaves)
    ok &= component_phi(mem(a->big_g) + (size_t)k * K * K, mem(a->big_row) + k * K, jg, face, lam);
  for (int k = kThreads - 1 - tid; k < n_one; k += kThreads) {
    const int r = mem(a->one_row)[k];
    double l = 0.0;
    if (face[r]) {
      const double g = mem(a->one_g)[k], d = sqrt(g);
      ok &= g > 0.0;
      l = -jg[r] / d / d;
    }
    lam[r] = l;
  }
  if (!ok) sh->fail = 1;
  __syncthreads();
}

// out = P(v) (GeneralConProjector::project, MPRGPProjection.h:412-431)
__device__ __noinline__ void project(Args *a_, Shared *sh, const double *v, double *out) {
  Args *a = uniform(a_);
  j_mul(a, v, a->j1, nullptr, nullptr);
  __syncthreads();
  multipliers(a, sh, false);
  const int n = a->n;
  for (int i = threadIdx.x; i < n; i += kThreads) mem(out)[i] = mem(v)[i] + jt_row(a, a->lam, i);
  __syncthreads();
}

// The face at v (DECIDE_FACE, :485-520) and PHI's multipliers at g.
__device__ __noinline__ void face_phi(Args *a_, Shared *sh, const double *v) {
  Args *a = uniform(a_);
  const int m = a->m;
  for (int i = threadIdx.x; i < m; i += kThreads) {
    const double jv = j_row(a, v, i);
    mem(a->j2)[i] = j_row(a, a->g, i);
    mem(a->face)[i] = fabs(jv - mem(a->c)[i]) < kEps ? 1 : 0;
  }
  __syncthreads();
  phi_multipliers(a, sh);
}

// The loop head's second half at x: BETA (:452-473) and the projection of
// t2 = x - alpha_bar phi (:474-484) from J of both (j1, j2), A p, and the sums
// |phi + beta|^2, beta.beta, (x - P(t2)).phi, p.A p, z.g.
__device__ __noinline__ void head(Args *a_, Shared *sh) {
  Args *a = uniform(a_);
  multipliers(a, sh, true);
  const int n = a->n;
  const auto beta = mem(a->beta), t2 = mem(a->t2), phi = mem(a->phi), x = mem(a->x), p = mem(a->p), ap = mem(a->ap);
  const auto z = mem(a->z), g = mem(a->g);
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const double tb = jt_row(a, a->lam, i), tp = jt_row(a, a->lam2, i), b0 = beta[i], t0 = t2[i];
    beta[i] = b0 - tb;
    t2[i] = t0 + tp;
  }
  product(a, sh, a->p, a->ap, nullptr);
  sums<5>(a, sh, 0, [&](int i, double *s) {
    const double gp = phi[i] + beta[i];
    s[0] = gp * gp;
    s[1] = beta[i] * beta[i];
    s[2] = (x[i] - t2[i]) * phi[i];
    s[3] = p[i] * ap[i];
    s[4] = z[i] * g[i];
  });
}

// isFeasible(y) (:298-310)
__device__ __noinline__ void feasible(Args *a_, Shared *sh) {
  Args *a = uniform(a_);
  const int m = a->m;
  if (threadIdx.x == 0) sh->infeasible = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += kThreads)
    if (j_row(a, a->y, i) < mem(a->c)[i] - kEps) sh->infeasible = 1;
  __syncthreads();
}

}  // namespace

__global__ void __launch_bounds__(kThreads) general_loop(const GenArgs *args) {
  __shared__ Block block;
  Shared *sh = (Shared *)&block;
  Args *a = (Args *)args;
  const int tid = threadIdx.x, n = a->n, max_it = a->max_it;
  const double ab = a->alpha_bar, tol = a->tol;
  double *x_ = a->x, *y_ = a->y, *g_ = a->g, *p_ = a->p, *z_ = a->z, *beta_ = a->beta;
  double *ap_ = a->ap, *t_ = a->t, *t2_ = a->t2;
  const auto x = mem(x_), y = mem(y_), g = mem(g_), p = mem(p_), z = mem(z_), phi = mem(a->phi);
  const auto beta = mem(beta_), ap = mem(ap_), t = mem(t_), t2 = mem(t2_);
  const bool pre = a->pre;
  const auto st = mem(a->st);
  double residual = st->residual, alpha = st->alpha, fx = st->fx, fy = st->fy;
  int iteration = st->iteration, num_cg = st->num_cg, num_exp = st->num_exp, num_prop = st->num_prop;
  int prop = st->prop, y_set = st->y_set, done = 0;
  int ax_set = st->ax_set;  // ax holds A x: an expansion's last product, which the next CG entry reads again
  bool in_cg = st->in_cg;
  const int stop = iteration + a->chunk;
  if (tid == 0) block.fail = block.spec = block.infeasible = 0;
  __syncthreads();
  auto result = [&] {  // the head's residual and proportional (:174-181), gamma = 1
    residual = sqrt(block.sum[0]);
    const double v2 = block.sum[2] * (1.0 / ab);
    prop = block.sum[1] <= (v2 > 0.0 ? v2 : 0.0);
  };
  while (true) {
    if (!in_cg) {  // the outer loop's head (:417-430)
      done = iteration >= max_it;
      if (done || iteration >= stop) break;
      for (int i = tid; i < n; i += kThreads) {
        beta[i] = g[i] - phi[i];
        t2[i] = x[i] + -ab * phi[i];
      }
      __syncthreads();
      j_mul(a, beta_, a->j1, t2_, a->j2);
      __syncthreads();
      head(a, sh);
      result();
      done = residual <= tol;
      if (done || block.fail || block.spec) break;
      if (prop) {  // CGMonotonicStep's entry (:272-284)
        alpha = block.sum[4] / block.sum[3];
        for (int i = tid; i < n; i += kThreads) y[i] = x[i] + -alpha * p[i];
        y_set = 1;
        __syncthreads();
        project(a, sh, y_, t_);
        product(a, sh, t_, a->t3, nullptr);
        if (!ax_set) product(a, sh, x_, a->ax, nullptr);
        dots(a, sh, 0, t_, a->t3, t_, a->b);
        dots(a, sh, 2, x_, a->ax, x_, a->b);
        fy = 0.5 * block.sum[0] - block.sum[1];
        fx = 0.5 * block.sum[2] - block.sum[3];
        in_cg = true;
      }
    }
    if (in_cg) {  // its steps (:285-309)
      while (prop && residual > tol && fy <= fx && iteration < max_it && iteration < stop) {
        ax_set = 0;
        for (int i = tid; i < n; i += kThreads) {
          x[i] = y[i];
          g[i] = g[i] + -alpha * ap[i];
        }
        __syncthreads();
        j_mul(a, g_, a->j2, nullptr, nullptr);
        __syncthreads();
        phi_multipliers(a, sh);
        for (int i = tid; i < n; i += kThreads) {
          const double f = g[i] + jt_row(a, a->lam, i);
          phi[i] = f;
          z[i] = pre ? f * mem(a->dinv)[i] : f;
          beta[i] = g[i] - f;
          t2[i] = x[i] + -ab * f;
        }
        __syncthreads();
        j_mul(a, beta_, a->j1, t2_, a->j2);
        dots(a, sh, 0, z_, ap_, p_, ap_);
        const double be = block.sum[0] / block.sum[1];
        for (int i = tid; i < n; i += kThreads) p[i] = z[i] + -be * p[i];
        head(a, sh);  // has barriers before p's neighbours are read
        result();
        if (block.fail || block.spec) break;
        alpha = block.sum[4] / block.sum[3];
        for (int i = tid; i < n; i += kThreads) y[i] = x[i] + -alpha * p[i];
        fx = fy;
        __syncthreads();
        project(a, sh, y_, t_);
        product(a, sh, t_, a->t3, nullptr);
        dots(a, sh, 0, t_, a->t3, t_, a->b);
        fy = 0.5 * block.sum[0] - block.sum[1];
        num_cg++;
        iteration++;
      }
      if (block.fail || block.spec) break;
      if (prop && residual > tol && fy <= fx && iteration < max_it) break;  // the launch's share is done
      in_cg = false;
      done = residual <= tol;
      if (done) break;
    }
    if (!prop && y_set) feasible(a, sh);
    if (prop || !y_set || block.infeasible) {  // ExpMonotonicStep (:250-271)
      num_exp++;
      project(a, sh, x_, y_);
      y_set = 1;
      product(a, sh, y_, a->ax, g_);
      face_phi(a, sh, y_);
      for (int i = tid; i < n; i += kThreads) {
        const double f = g[i] + jt_row(a, a->lam, i);
        phi[i] = f;
        y[i] = y[i] + -ab * f;
      }
      __syncthreads();
      project(a, sh, y_, x_);
      product(a, sh, x_, a->ax, g_);
      ax_set = 1;
      __syncthreads();
    } else {  // g = A x - b, then PropStep (:219-243, 435-437)
      num_prop++;
      product(a, sh, x_, a->ax, g_);
      product(a, sh, beta_, ap_, nullptr);
      ax_set = 0;
      __syncthreads();
      dots(a, sh, 0, beta_, ap_, g_, beta_);
      const double al = block.sum[1] / block.sum[0];
      for (int i = tid; i < n; i += kThreads) {
        t[i] = x[i] + -al * beta[i];
        g[i] = g[i] + -al * ap[i];
      }
      __syncthreads();
      project(a, sh, t_, x_);
    }
    face_phi(a, sh, x_);
    for (int i = tid; i < n; i += kThreads) {
      const double f = g[i] + jt_row(a, a->lam, i), zz = pre ? f * mem(a->dinv)[i] : f;
      phi[i] = f;
      z[i] = zz;
      p[i] = zz;
    }
    __syncthreads();
    iteration++;
  }
  __syncthreads();
  if (tid == 0) {
    st->residual = residual;
    st->alpha = alpha;
    st->fx = fx;
    st->fy = fy;
    st->iteration = iteration;
    st->num_cg = num_cg;
    st->num_exp = num_exp;
    st->num_prop = num_prop;
    st->prop = prop;
    st->y_set = y_set;
    st->ax_set = ax_set;
    st->in_cg = in_cg;
    st->done = done;
    st->fail = block.fail || (block.spec && !done);
  }
}

hipError_t launch_general_loop(hipStream_t s, const GenArgs *args) {
  general_loop<<<1, kThreads, 0, s>>>(args);
  return hipGetLastError();
}

}  // namespace mprgp
