// hmv_construct.hip -- the H-matrix fill on the device: dense leaves by entry
// evaluation, low-rank leaves by ACA+, and the arena fill from device
// factors.
//
// The reference fills its leaves on the CPU (HACApK_generate,
// m_HACApK_base.f90:1005-1051: HACApK_acaplus per admissible block,
// :783-975, and the entry function HACApK_entry_ij per dense entry).  Here
// the host keeps the cluster tree and the block list (cheap), and the device
// evaluates every entry and runs every block's ACA+ in parallel: one
// workgroup per block, all of its lanes on the block's rows/columns, the
// scalar steps of ACA+ in the same order and arithmetic as the host
// restatement (the cross updates, the pivot searches with their first-index
// ties).  Only the norms are summed in another order; they are compared with
// thresholds, and a block with one too near its threshold for the order not to
// matter runs again with all of them in the host's, so where the entries are
// the host's (the centroid kernel off the diagonal) ranks and factors are too.
// Floating-point contraction is off in this file, so entries and updates round
// as the host's do.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "hmv.h"
#include "hmv_engine.h"
#include "hmv_internal.h"
#include "hmv_plan.h"

#pragma clang fp contract(off)

namespace {

constexpr int kT = 256;
// Factor columns reserved per block in the first pass: ranks grow with the
// digits asked for (at 163,840 unknowns at most 16 for 1e-5, 14 for 1e-4); a
// block that needs more runs again with its full bound.
int first_columns(double eps) {
  const double digits = eps > 0.0 && eps < 1.0 ? std::ceil(-std::log10(eps)) : 0.0;
  return std::max(16, std::min(64, 10 + 3 * (int)std::min(digits, 100.0)));
}
// Bytes of reserved columns in use at a time.  The blocks run in batches of
// this size and each batch's factors are packed behind it, so that a
// construction allocates little more than the factors: memory given back is
// cleared at some 40 GB/s before it can be had again, and with 64 columns for
// every block at once (7.2 GB at 81,920 unknowns for 0.9 GB of factors) every
// few constructions waited 0.3 to 3 s for it.
constexpr size_t kAcaBatchBytes = (size_t)1 << 30;

// ---- entry function --------------------------------------------------------

// m_ppohBEM_user_func.f90:42-43 (default-REAL literals in REAL(8) parameters)
__device__ constexpr double kPiF = (double)3.141592653589793f;
__device__ constexpr double kEps0F = (double)8.854187818f * 1e-12;
constexpr int kKernelPpohbem = 0;
constexpr int kKernelCentroid = 1;

struct Geo {
  const double *cent;   // nface x 3, original order
  const double *area;   // nface
  const double *nodes;  // nnode x 3
  const int *faces;     // nface x 3, 0-based
  const int *lod;       // cluster order -> original (1-based)
  int kernel;
};

__device__ inline void cross3(const double u[3], const double v[3], double w[3]) {
  w[0] = u[1] * v[2] - u[2] * v[1];
  w[1] = u[2] * v[0] - u[0] * v[2];
  w[2] = u[0] * v[1] - u[1] * v[0];
}
__device__ inline double dot3(const double a[3], const double b[3]) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// Signed sum of the analytic 1/r potential of a flat triangle at (x,y,z),
// face_integral (m_ppohBEM_user_func.f90:49-100) term by term.
__device__ double triangle_potential_sum(const double xs[3], const double ys[3],
                                         const double zs[3], double x, double y, double z) {
  double r[3];
  for (int i = 0; i < 3; ++i) {
    const double dx = xs[i] - x, dy = ys[i] - y, dz = zs[i] - z;
    r[i] = sqrt(dx * dx + dy * dy + dz * dz);
  }
  double u[3] = {xs[1] - xs[0], ys[1] - ys[0], zs[1] - zs[0]};
  double v[3] = {xs[2] - xs[1], ys[2] - ys[1], zs[2] - zs[1]};
  double w[3];
  cross3(u, v, w);
  const double wn = sqrt(dot3(w, w));
  w[0] /= wn;
  w[1] /= wn;
  w[2] /= wn;
  u[0] = x - xs[0];
  u[1] = y - ys[0];
  u[2] = z - zs[0];
  const double zp = dot3(u, w);
  const double ox = x - zp * w[0], oy = y - zp * w[1], oz = z - zp * w[2];
  const double zpabs = fabs(zp);
  double sum = 0.0;
  for (int i = 0; i < 3; ++i) {
    const int j = (i + 1) % 3;
    u[0] = xs[j] - ox;
    u[1] = ys[j] - oy;
    u[2] = zs[j] - oz;
    const double xj = sqrt(dot3(u, u));
    u[0] /= xj;
    u[1] /= xj;
    u[2] /= xj;
    cross3(w, u, v);
    const double xi = (xs[i] - ox) * u[0] + (ys[i] - oy) * u[1] + (zs[i] - oz) * u[2];
    const double yi = (xs[i] - ox) * v[0] + (ys[i] - oy) * v[1] + (zs[i] - oz) * v[2];
    const double dx = xj - xi, dy = -yi;
    const double t = sqrt(dx * dx + dy * dy);
    const double l = dx / t, m = dy / t;
    const double d = l * yi - m * xi;
    const double ti = l * xi + m * yi, tj = l * xj;
    const double theta = atan2(yi, xi);
    const double omega = theta - atan2(r[i] * d, zpabs * ti) + atan2(r[j] * d, zpabs * tj);
    const double q = log((r[j] + tj) / (r[i] + ti));
    const double g = d * q - zpabs * omega;
    sum = sum + g;
  }
  return sum;
}

// The centroid kernel off the diagonal (0-based faces).
__device__ inline double centroid_entry(const Geo &g, int fi, int fj) {
  const double dx = g.cent[3 * fi] - g.cent[3 * fj];
  const double dy = g.cent[3 * fi + 1] - g.cent[3 * fj + 1];
  const double dz = g.cent[3 * fi + 2] - g.cent[3 * fj + 2];
  return g.area[fj] / (4.0 * M_PI * sqrt(dx * dx + dy * dy + dz * dz));
}

// HACApK_entry_ij(i, j) for 1-based original indices: collocation at the
// centroid of face i, source face j (m_ppohBEM_matrix_element_ij.f90:49-76).
__device__ double entry(const Geo &g, int i, int j) {
  const int fi = i - 1, fj = j - 1;
  if (g.kernel == kKernelCentroid && fi != fj) return centroid_entry(g, fi, fj);
  double xs[3], ys[3], zs[3];
  for (int a = 0; a < 3; ++a) {
    const int nn = g.faces[3 * fj + a];
    xs[a] = g.nodes[3 * nn];
    ys[a] = g.nodes[3 * nn + 1];
    zs[a] = g.nodes[3 * nn + 2];
  }
  const double s =
      triangle_potential_sum(xs, ys, zs, g.cent[3 * fi], g.cent[3 * fi + 1], g.cent[3 * fi + 2]);
  if (g.kernel == kKernelPpohbem) return fabs(s) / (4.0 * kPiF * kEps0F);
  return fabs(s) / (4.0 * M_PI);
}

// ---- leaves ----------------------------------------------------------------

struct CLeaf {
  int ltmtx, nstrtl, ndl, nstrtt, ndt;
  int cap;        // low rank: factor columns held (reserved) at base
  double *base;   // dense: A (ndl rows of ndt); low rank: V (ndt x cap), then U (ndl x cap)
  double *pa;     // low rank scratch: reference column (ndl), then reference row (ndt)
  int *msk;       // low rank scratch: row mask (ndl), then column mask (ndt)
};

struct AcaParams {
  double eps, eps_factor;
  int kmax, kmin;
};

enum { kAcaOk = 0, kAcaOverflow = 1, kAcaNear = 2 };

__global__ __launch_bounds__(kT) void k_dense(const CLeaf *__restrict__ lv, Geo g) {
  const CLeaf L = lv[blockIdx.x];
  const int64_t n = (int64_t)L.ndl * L.ndt;
  for (int64_t e = threadIdx.x; e < n; e += kT) {
    const int il = (int)(e / L.ndt), it = (int)(e % L.ndt);
    L.base[e] = entry(g, g.lod[L.nstrtl - 1 + il], g.lod[L.nstrtt - 1 + it]);
  }
}

// ACA+ runs one workgroup per block.  Its scalar steps are sequential and
// every vector pass of a step ends in a reduction that the next one needs, so
// a block's time is its passes: their memory round trips for a short block,
// its vectors over the workgroup's lanes for a long one.  Hence
//  - one wave for short blocks (reductions by lane shuffles; most blocks are
//    short, and many run at once), NT = 256 or 1024 threads for longer ones
//    (aca_class);
//  - three passes a step: the pivot column or row with its largest entry, the
//    other one with the scaling and the update of its reference vector, the
//    update of the other reference vector; each also forms the norms and the
//    largest entries that the step reads from what it just wrote.
// 163,840 unknowns, two spheres (blocks up to 41,088 x 41,088): 173 ms with
// one wave per block and a pass per operation, 9.1 ms now; one sphere of
// 81,920: 21.4 ms, 3.9 ms now; the factors are the same bits.

// A value that is the same in every lane, in scalar registers.
__device__ inline double uniform(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Largest |entry| with its first index, and the sum of squares, of the
// entries one thread has seen (HACApK_maxabsvalloc_d, HACApK_unrm_d).
// Entries below 1e-30 do not count in the norm, as there.
struct VecStat {
  double mx = 0.0;
  int ix = -1;  // none yet
  double ss = 0.0;
  __device__ void add(double v, int a) {
    const double x = fabs(v);
    if (ix < 0 || x > mx) {
      mx = x;
      ix = a;
    }
    if (!(x < 1.0e-30)) ss = ss + x * x;
  }
  __device__ void merge(double omx, int oix, double oss) {
    if (oix >= 0 && (ix < 0 || omx > mx || (omx == mx && oix < ix))) {
      mx = omx;
      ix = oix;
    }
    ss = ss + oss;
  }
};

// LDS of a workgroup's reductions: two buffers in turn, so that one barrier
// per reduction is enough (a buffer is written again only after the next
// reduction's barrier, which every reader has passed).
template <int NT>
struct AcaShared {
  double mx[2][2][NT / 64], ss[2][2][NT / 64];
  int ix[2][2][NT / 64];
};

// Reductions over the workgroup; every thread gets the same values, and the
// barrier makes what the threads wrote before it visible to all of them.
template <int NT>
struct Aca {
  AcaShared<NT> &sh;
  int turn = 0;
  __device__ explicit Aca(AcaShared<NT> &s) : sh(s) {}

  __device__ static void wave_merge(VecStat &s, int from = 32) {
#pragma unroll 1
    for (int off = from; off > 0; off >>= 1) {
      const double omx = __shfl_xor(s.mx, off, 64), oss = __shfl_xor(s.ss, off, 64);
      const int oix = __shfl_xor(s.ix, off, 64);
      s.merge(omx, oix, oss);
    }
    settle(s);
  }
  // the first lane's statistics (with entries that are no numbers the lanes
  // may disagree), in scalar registers
  __device__ static void settle(VecStat &s) {
    s.mx = uniform(s.mx);
    s.ss = uniform(s.ss);
    s.ix = __builtin_amdgcn_readfirstlane(s.ix);
  }
  // the waves' statistics of this turn, merged by every wave alike
  __device__ void gather(VecStat &s, int which) {
    const int v = threadIdx.x & (NT / 64 - 1);
    s.mx = sh.mx[turn][which][v];
    s.ss = sh.ss[turn][which][v];
    s.ix = sh.ix[turn][which][v];
    wave_merge(s, NT / 128);
  }
  // Two statistics at once (`both`), or one.
  __device__ void reduce(VecStat &p, VecStat &q, bool both) {
    wave_merge(p);
    if (both) wave_merge(q);
    if constexpr (NT > 64) {
      const int w = threadIdx.x >> 6;
      if ((threadIdx.x & 63) == 0) {
        sh.mx[turn][0][w] = p.mx;
        sh.ss[turn][0][w] = p.ss;
        sh.ix[turn][0][w] = p.ix;
        if (both) {
          sh.mx[turn][1][w] = q.mx;
          sh.ss[turn][1][w] = q.ss;
          sh.ix[turn][1][w] = q.ix;
        }
      }
      __syncthreads();
      gather(p, 0);
      if (both) gather(q, 1);
      turn ^= 1;
    } else {
      __syncthreads();
    }
  }
  __device__ void reduce(VecStat &p) {
    VecStat none;
    reduce(p, none, false);
  }
  // ||vec|| from its statistics.  The squares are safe up to 1e150; past
  // that the entries are scaled by the largest.  The reference accumulates in
  // entry order; here the order is the reduction's, which moves the last bits
  // of a number that is only compared with thresholds (see far).
  __device__ double norm(const VecStat &s, const double *vec, int n) {
    if (!(s.mx > 1.0e150)) return sqrt(s.ss);
    VecStat t;
    for (int a = threadIdx.x; a < n; a += NT) t.add(vec[a] / s.mx, a);
    reduce(t);
    return s.mx * sqrt(t.ss);
  }
};

// Two sums of n squares differ by less than n 2^-52 in their norm: 4e-9 at 16
// million entries.  A norm at least kNear from a threshold (relative to it)
// lies on the same side of it in every order of summation.
constexpr double kNear = 1.0e-8;
__device__ inline bool far(double v, double thr) {
  // not with an infinity or a NaN
  return fabs(v - thr) > kNear * thr || (v == 0.0 && thr == 0.0);
}

// HACApK_unrm_d, bit for bit, in one wave.  Its running scale zscl is the
// prefix maximum of the |entries| (those below 1e-30 skipped): each lane forms
// its entry's ratio zscl/zza or zza/zscl from a prefix maximum over the wave,
// and only the accumulation of zzz runs entry by entry.
__device__ double unrm(const double *vec, int n) {
  const int lane = threadIdx.x;
  double zscl = 0.0, zzz = 1.0;  // the same in every lane
#pragma unroll 1
  for (int c0 = 0; c0 < n; c0 += 64) {
    const int nl = min(64, n - c0);
    const double a = lane < nl ? fabs(vec[c0 + lane]) : 0.0;
    const bool skip = lane >= nl || a < 1.0e-30;
    double incl = skip ? 0.0 : a;
#pragma unroll 1
    for (int off = 1; off < 64; off <<= 1) {
      const double o = __shfl_up(incl, off, 64);
      if (lane >= off && o > incl) incl = o;
    }
    const double before = __shfl_up(incl, 1, 64);
    const double m = lane > 0 && before > zscl ? before : zscl;  // zscl before the entry
    const bool grows = !skip && m < a;
    const double q = skip ? 0.0 : grows ? m / a : a / m;
    const unsigned long long g = __ballot(grows), none = __ballot(skip);
#pragma unroll 1
    for (int l = 0; l < nl; ++l) {
      if ((none >> l) & 1ull) continue;
      const double ql = __shfl(q, l, 64);
      if ((g >> l) & 1ull)
        zzz = 1.0 + zzz * ql * ql;
      else
        zzz = zzz + ql * ql;
    }
    const double most = __shfl(incl, nl - 1, 64);
    if (most > zscl) zscl = most;
  }
  return uniform(zscl * sqrt(zzz));
}

// Entry a of the residual column ip (col) or row ip of a block after k
// crosses (HACApK_calc_vec): the matrix entry minus the cross products
// (summed in cross order before the subtraction); zero at a masked position
// (there are none before the first cross).
template <bool CENT>
__device__ inline double residual(const CLeaf &L, const Geo &g, bool col, int k, int ip, int a,
                                  const double *U, const double *V) {
  if (L.msk[col ? a : L.ndl + a] != 0) return 0.0;
  const int i = g.lod[col ? a + L.nstrtl - 1 : ip + L.nstrtl - 2];
  const int j = g.lod[col ? ip + L.nstrtt - 2 : a + L.nstrtt - 1];
  const double e = CENT ? centroid_entry(g, i - 1, j - 1) : entry(g, i, j);
  if (k == 0) return e;
  const int sx = col ? L.ndl : L.ndt, sy = col ? L.ndt : L.ndl;
  const double *px = (col ? U : V) + a, *py = (col ? V : U) + (ip - 1);
  double t = 0.0;
  int it = 0;
#pragma unroll 1
  for (; it + 4 <= k; it += 4) {  // four crosses' loads together
    double x[4], y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      x[q] = px[(size_t)(it + q) * sx];
      y[q] = py[(size_t)(it + q) * sy];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) t = t + x[q] * y[q];
  }
#pragma unroll 1
  for (; it < k; ++it) t = t + px[(size_t)it * sx] * py[(size_t)it * sy];
  return e - t;
}

// A thread's entries tid, tid + nt, ... of that column or row into vec, with
// their statistics.
template <bool CENT>
__device__ inline VecStat residual_loop(const CLeaf &L, const Geo &g, bool col, int k, int ip,
                                        double *vec, const double *U, const double *V, int nt) {
  VecStat s;
  const int n = col ? L.ndl : L.ndt;
#pragma unroll 1
  for (int a = threadIdx.x; a < n; a += nt) {
    const double e = residual<CENT>(L, g, col, k, ip, a, U, V);
    vec[a] = e;
    s.add(e, a);
  }
  return s;
}
// With the analytic entry, a call of its own: one copy of that code.
__device__ __attribute__((noinline)) VecStat residual_any(const CLeaf &L, const Geo &g, bool col,
                                                          int k, int ip, double *vec,
                                                          const double *U, const double *V,
                                                          int nt) {
  return residual_loop<false>(L, g, col, k, ip, vec, U, V, nt);
}
template <bool CENT>
__device__ inline VecStat residual_part(const CLeaf &L, const Geo &g, bool col, int k, int ip,
                                        double *vec, const double *U, const double *V, int nt) {
  if constexpr (CENT)
    return residual_loop<true>(L, g, col, k, ip, vec, U, V, nt);
  else
    return residual_any(L, g, col, k, ip, vec, U, V, nt);
}

// HACApK_acaplus (m_HACApK_base.f90:783-975) with param(61) = 1, for one
// block per workgroup; restates the host fill's ACA+ step for step.  CENT:
// the centroid kernel on blocks that hold no diagonal entry.  HOST: norms in
// the host's order (NT = 64); without it a block with a norm not far from its
// threshold ends as kAcaNear, a matter of chance in 1e-8 per test.  (Forming
// that norm here instead costs the others 5% (1,024 threads) to 36% (one
// wave): registers held for a call that hardly ever comes.)
template <int NT, bool CENT, bool HOST>
__global__ __launch_bounds__(NT) void k_aca(const CLeaf *__restrict__ lv, Geo g, AcaParams p,
                                            int *__restrict__ kt_out, int *__restrict__ status) {
  __shared__ AcaShared<NT> shared;
  Aca<NT> R(shared);
  const int id = blockIdx.x;
  const CLeaf L = lv[id];
  const int ndl = L.ndl, ndt = L.ndt, cap = L.cap, tid = threadIdx.x;
  double *V = L.base;                    // zab(ndt, cap)
  double *U = L.base + (size_t)ndt * cap;  // zaa(ndl, cap)
  double *pa_ref = L.pa, *pb_ref = L.pa + ndl;
  int *lrow_msk = L.msk, *lcol_msk = L.msk + ndl;

  for (int a = tid; a < ndl + ndt; a += NT) L.msk[a] = 0;
  __syncthreads();

  const double eps = p.eps;
  const double ACA_EPS = p.eps_factor * eps;
  const double za_ACA_EPS = (double)1.0e-30f;
  const double piv_min = (double)1.0e-20f;
  int ntries = max(ndl, ndt) + 1, ntries_row = 6, ntries_col = 6;
  int k = 0;
  int st = kAcaOk;

  // the residual column (row) ip after kk crosses into vec, with its statistics
  auto calc = [&](bool col, int kk, int ip, double *vec) {
    VecStat s = residual_part<CENT>(L, g, col, kk, ip, vec, U, V, NT);
    R.reduce(s);
    return s;
  };
  // y += x s, with y's statistics
  auto axpy = [&](double *y, const double *x, int n, double s) {
    VecStat t;
    for (int a = tid; a < n; a += NT) {
      const double v = y[a] + x[a] * s;
      y[a] = v;
      t.add(v, a);
    }
    R.reduce(t);
    return t;
  };
  auto set_mask = [&](int *m, int i1) {
    if (tid == 0) m[i1 - 1] = 1;
  };

  auto norm = [&](const VecStat &s, const double *vec, int n) {
    if constexpr (HOST)
      return unrm(vec, n);
    else
      return R.norm(s, vec, n);
  };
  // whether a norm lies below thr
  auto below = [&](double v, double thr) {
    if constexpr (!HOST)
      if (!far(v, thr)) st = kAcaNear;
    return v < thr;
  };

  int j_ref = 1;
  VecStat sa = calc(true, k, j_ref, pa_ref);  // of pa_ref, as it is now
  double colnorm = norm(sa, pa_ref, ndl);
  int i_ref;
  {
    // first index of the smallest |entry|: the largest of their negatives
    VecStat s;
    for (int a = tid; a < ndl; a += NT) {
      const double x = fabs(pa_ref[a]);
      if (s.ix < 0 || x < -s.mx) {
        s.mx = -x;
        s.ix = a;
      }
    }
    R.reduce(s);
    i_ref = s.ix + 1;
  }
  VecStat sb = calc(false, k, i_ref, pb_ref);  // of pb_ref, as it is now
  double rownorm = norm(sb, pb_ref, ndt);

  double apxnorm = 0.0;
  int lstop_aca = 0;
  int i = 0, j = 0;
  while ((k < p.kmax) && (ntries_row > 0 || ntries_col > 0) && (ntries > 0)) {
    ntries = ntries - 1;
    if (k + 1 > cap) {
      st = kAcaOverflow;
      break;
    }
    double *pcol = U + (size_t)k * ndl;
    double *prow = V + (size_t)k * ndt;
    i = sa.ix + 1;
    j = sb.ix + 1;
    // The cross: the reference vector with the larger entry gives the first
    // of column j and row i (its own copy when that is the reference's), its
    // largest entry the pivot and the other index; the first is scaled by
    // the pivot.  Then pb_ref -= prow pcol(i_ref), pa_ref -= pcol prow(j_ref).
    const bool colfirst = sb.mx > sa.mx;
    const int n1 = colfirst ? ndl : ndt, n2 = colfirst ? ndt : ndl;
    double *v1 = colfirst ? pcol : prow, *v2 = colfirst ? prow : pcol;
    VecStat s1;
    if (colfirst ? j != j_ref : i != i_ref) {
      s1 = calc(colfirst, k, colfirst ? j : i, v1);
    } else {
      const double *src = colfirst ? pa_ref : pb_ref;
      for (int a = tid; a < n1; a += NT) v1[a] = src[a];
      s1 = colfirst ? sa : sb;
      __syncthreads();
    }
    if (colfirst)
      i = s1.ix + 1;
    else
      j = s1.ix + 1;
    VecStat q1, q2;  // of the scaled v1 and of v2 (norms)
    bool a_done = false, b_done = false;
    if (s1.mx < ACA_EPS && k >= p.kmin) {
      lstop_aca = 1;
      // the other one is not formed; the step may still count it (below), as
      // zeros
      for (int a = tid; a < n2; a += NT) v2[a] = 0.0;
    } else {
      // entries of v1 that other threads are about to scale
      const double piv = uniform(v1[(colfirst ? i : j) - 1]);
      const double at_ref = uniform(v1[(colfirst ? i_ref : j_ref) - 1]);
      __syncthreads();
      if (!(fabs(piv) > piv_min)) {
        k = max(k - 1, 0);
        break;
      }
      const double inv = 1.0 / piv;
      // v2 and, when its reference vector is another one, that vector's
      // update by v2 times the scaled v1's entry at the reference
      const bool upd = colfirst ? i != i_ref : j != j_ref;
      const double zinv = -(at_ref * inv);
      double *ref2 = colfirst ? pb_ref : pa_ref;
      VecStat sr;
      q2 = residual_part<CENT>(L, g, !colfirst, k, colfirst ? i : j, v2, U, V, NT);
      if (upd)
        for (int a = tid; a < n2; a += NT) {
          const double v = ref2[a] + v2[a] * zinv;
          ref2[a] = v;
          sr.add(v, a);
        }
      for (int a = tid; a < n1; a += NT) {
        const double e = v1[a] * inv;
        v1[a] = e;
        q1.add(e, a);
      }
      R.reduce(q1, q2, true);
      if (upd) {
        R.reduce(sr);
        if (colfirst) {
          sb = sr;
          b_done = true;
        } else {
          sa = sr;
          a_done = true;
        }
      }
    }
    set_mask(lrow_msk, i);
    set_mask(lcol_msk, j);
    __syncthreads();

    if (i != i_ref) {
      if (!b_done) sb = axpy(pb_ref, prow, ndt, -uniform(pcol[i_ref - 1]));
      rownorm = norm(sb, pb_ref, ndt);
    }
    if (i == i_ref || below(rownorm, ACA_EPS)) {
      if (i == i_ref) ntries_row = ntries_row + 1;
      if (ntries_row > 0) {
        rownorm = 0.0;
        i = i_ref;
        while (i != ((i_ref + ndl - 2) % ndl) + 1 && below(rownorm, za_ACA_EPS) && ntries_row > 0) {
          if (__builtin_amdgcn_readfirstlane(lrow_msk[i - 1]) == 0) {
            if (k + 1 > cap) {
              st = kAcaOverflow;
              break;
            }
            sb = calc(false, k + 1, i, pb_ref);
            rownorm = norm(sb, pb_ref, ndt);
            if (below(rownorm, ACA_EPS)) set_mask(lrow_msk, i);
            __syncthreads();
            ntries_row = ntries_row - 1;
          } else {
            rownorm = 0.0;
          }
          i = (i % ndl) + 1;
        }
        if (st != kAcaOk) break;
        i_ref = ((i + ndl - 2) % ndl) + 1;
      }
    }

    if (j != j_ref) {
      if (!a_done) sa = axpy(pa_ref, pcol, ndl, -uniform(prow[j_ref - 1]));
      colnorm = norm(sa, pa_ref, ndl);
    }
    if (j == j_ref || below(colnorm, ACA_EPS)) {
      if (j == j_ref) ntries_col = ntries_col + 1;
      if (ntries_col > 0) {
        colnorm = 0.0;
        j = j_ref;
        while (j != ((j_ref + ndt - 2) % ndt) + 1 && below(colnorm, za_ACA_EPS) && ntries_col > 0) {
          if (__builtin_amdgcn_readfirstlane(lcol_msk[j - 1]) == 0) {
            if (k + 1 > cap) {
              st = kAcaOverflow;
              break;
            }
            sa = calc(true, k + 1, j, pa_ref);
            colnorm = norm(sa, pa_ref, ndl);
            if (below(colnorm, ACA_EPS)) set_mask(lcol_msk, j);
            __syncthreads();
            ntries_col = ntries_col - 1;
          } else {
            colnorm = 0.0;
          }
          j = (j % ndt) + 1;
        }
        if (st != kAcaOk) break;
        j_ref = ((j + ndt - 2) % ndt) + 1;
      }
    }

    if (below(colnorm, ACA_EPS) && below(rownorm, ACA_EPS) && k >= p.kmin) {
      lstop_aca = 1;
      k = k + 1;
    }
    if (lstop_aca == 0) {
      const double blknorm = norm(q1, v1, n1) * norm(q2, v2, n2);
      if (k == 0) {
        apxnorm = blknorm;
      } else {
        const double thr = apxnorm * eps;
        const bool blk = below(blknorm, thr), row = below(rownorm, thr), col = below(colnorm, thr);
        if (blk && row && col && k >= p.kmin) lstop_aca = 1;
      }
    }
    if (st != kAcaOk || (lstop_aca == 1 && k >= p.kmin)) break;
    k = k + 1;
  }
  if (st == kAcaOk && k > cap) st = kAcaOverflow;
  if (tid == 0) {
    kt_out[id] = k;
    status[id] = st;
  }
}

// The kt factor columns of a block (V, then U) from its reserved columns to
// dst[blockIdx.x], V and U next to each other (null: none to copy); gridDim.y
// workgroups share a block.
__global__ __launch_bounds__(1024) void k_pack(const CLeaf *__restrict__ lv,
                                               const int *__restrict__ kt,
                                               double *const *__restrict__ dst) {
  const CLeaf L = lv[blockIdx.x];
  double *o = dst[blockIdx.x];
  if (!o) return;
  const int64_t k = kt[blockIdx.x], nv = k * L.ndt, nu = k * L.ndl;
  const double *u = L.base + (int64_t)L.ndt * L.cap;
  const int64_t t0 = blockIdx.y * (int64_t)blockDim.x + threadIdx.x;
  const int64_t step = (int64_t)gridDim.y * blockDim.x;
  for (int64_t e = t0; e < nv; e += step) o[e] = L.base[e];
  for (int64_t e = t0; e < nu; e += step) o[nv + e] = u[e];
}

// ---- arena fill from device factors ----------------------------------------

__device__ inline uint16_t to_bf16(double v) {
  const float f = (float)v;
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
  const uint32_t lsb = (u >> 16) & 1u;
  u += 0x7fffu + lsb;
  return (uint16_t)(u >> 16);
}

__global__ __launch_bounds__(kT) void k_fill(const HmvFillOp *__restrict__ ops, char *arena) {
  const HmvFillOp o = ops[blockIdx.x];
  const int64_t n = (int64_t)o.nrows * o.ncols;
  char *dst = arena + o.dst;
  for (int64_t e = threadIdx.x; e < n; e += kT) {
    const int r = (int)(e % o.nrows), c = (int)(e / o.nrows);
    const double v = o.src[r * o.s_r + c * o.s_c];
    const int64_t i = (o.r0 + r) + (int64_t)o.ld * (o.c0 + c);
    if (o.dt == HMV_DT_F64)
      reinterpret_cast<double *>(dst)[i] = v;
    else if (o.dt == HMV_DT_F32)
      reinterpret_cast<float *>(dst)[i] = (float)v;
    else
      reinterpret_cast<uint16_t *>(dst)[i] = to_bf16(v);
  }
}

}  // namespace

namespace hmv {

// Runs the arena fill records on the device (the image already zeroed).
hipError_t launch_fill(const FillOps &ops, char *arena) {
  constexpr size_t kBatch = 1 << 20;  // records per launch (grid size)
  HmvFillOp *d = nullptr;
  const size_t nb = std::min(ops.size(), kBatch);
  hipError_t e = hipMalloc((void **)&d, sizeof(HmvFillOp) * std::max<size_t>(1, nb));
  if (e != hipSuccess) return e;
  for (size_t o = 0; o < ops.size() && e == hipSuccess; o += kBatch) {
    const size_t n = std::min(kBatch, ops.size() - o);
    e = hipMemcpy(d, ops.data() + o, sizeof(HmvFillOp) * n, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_fill, dim3((unsigned)n), dim3(kT), 0, nullptr, d, arena);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
  }
  (void)hipFree(d);
  return e;
}

}  // namespace hmv

// ---- public object ---------------------------------------------------------

struct hmv_dleaves_s {
  int nd = 0, nlf = 0;
  std::vector<CLeaf> lv;           // host copy of the device leaf table
  std::vector<int> kt;             // per leaf
  std::vector<hmv::RefLeaf> rec;   // leaf records with device factor pointers
  std::vector<void *> allocs;      // device allocations to free
  double seconds = 0.0;            // device fill time
  ~hmv_dleaves_s() {
    for (void *p : allocs) (void)hipFree(p);
  }
};

namespace {

hipError_t dalloc(hmv_dleaves_s *d, void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, std::max<size_t>(bytes, 8));
  if (e == hipSuccess) d->allocs.push_back(*p);
  return e;
}

// Threads per block of ACA+, by the longer side: one wave up to kAcaShort
// entries (at most four per lane: the passes are round trips, and barriers
// between waves would only add to them), 256 threads up to kAcaLong, else
// 1024 (at 2,592 rows a block's 256 threads already make 11 trips a pass).
constexpr int kAcaShort = 256, kAcaLong = 2048;

template <int NT, bool CENT, bool HOST = false>
void launch_aca_class(int n, const CLeaf *d_lv, const Geo &g, const AcaParams &p, int *d_kt,
                      int *d_st) {
  if (n > 0)
    hipLaunchKernelGGL((k_aca<NT, CENT, HOST>), dim3((unsigned)n), dim3(NT), 0, nullptr, d_lv, g, p,
                       d_kt, d_st);
}
// The blocks of one batch, in the order of their classes (n of each).
template <bool CENT>
void launch_aca(const int (&n)[3], const CLeaf *d_lv, const Geo &g, const AcaParams &p, int *d_kt,
                int *d_st) {
  launch_aca_class<1024, CENT>(n[0], d_lv, g, p, d_kt, d_st);
  launch_aca_class<256, CENT>(n[1], d_lv + n[0], g, p, d_kt + n[0], d_st + n[0]);
  launch_aca_class<64, CENT>(n[2], d_lv + n[0] + n[1], g, p, d_kt + n[0] + n[1],
                             d_st + n[0] + n[1]);
}

int aca_class(const CLeaf &L) {
  const int len = std::max(L.ndl, L.ndt);
  return len > kAcaLong ? 0 : len > kAcaShort ? 1 : 2;
}

// Runs ACA+ on the listed low-rank leaves (longest first) with at most
// `columns` factor columns each, in batches; packs their factors into
// allocations of d, and sets their records' base and cap and d->kt.  `again`
// receives the leaves that need more columns, `near` those with a norm at its
// threshold (none with host_norms).
hipError_t run_aca(hmv_dleaves_s *d, const std::vector<int> &ids, const Geo &g,
                   const AcaParams &p, int columns, bool host_norms, std::vector<int> &again,
                   std::vector<int> &near) {
  if (ids.empty()) return hipSuccess;
  // the analytic entry is needed with its kernel and on a diagonal
  bool cent = g.kernel == kKernelCentroid;
  size_t most = 0, total = 0;  // bytes of the largest block and of all
  auto cap_of = [&](const CLeaf &L) {
    return std::min(columns, std::min(p.kmax, std::min(L.ndl, L.ndt)) + 1);
  };
  auto bytes_of = [&](const CLeaf &L) {
    return sizeof(double) * ((size_t)L.ndl + L.ndt) * (size_t)cap_of(L);
  };
  for (int i : ids) {
    const CLeaf &L = d->lv[i];
    cent = cent && (L.nstrtl + L.ndl <= L.nstrtt || L.nstrtt + L.ndt <= L.nstrtl);
    most = std::max(most, bytes_of(L));
    total += bytes_of(L);
  }
  const size_t limit = std::min(total, std::max(most, kAcaBatchBytes));
  // batches [first, last) of ids; the largest one's vectors and blocks
  std::vector<size_t> ends;
  size_t used = 0, len = 0, count = 0, len_most = 0, count_most = 0;
  for (size_t q = 0; q < ids.size(); ++q) {
    const CLeaf &L = d->lv[ids[q]];
    if (used > 0 && used + bytes_of(L) > limit) {
      ends.push_back(q);
      used = len = count = 0;
    }
    used += bytes_of(L);
    len += (size_t)L.ndl + L.ndt;
    ++count;
    len_most = std::max(len_most, len);
    count_most = std::max(count_most, count);
  }
  ends.push_back(ids.size());
  struct Buf {  // freed on every exit
    char *p = nullptr;
    ~Buf() { (void)hipFree(p); }
  } buf;
  const size_t o_pa = limit, o_lv = o_pa + sizeof(double) * len_most,
               o_dst = o_lv + sizeof(CLeaf) * count_most,
               o_msk = o_dst + sizeof(double *) * count_most,
               o_kt = o_msk + sizeof(int) * len_most, o_st = o_kt + sizeof(int) * count_most,
               bytes = o_st + sizeof(int) * count_most;
  hipError_t e = hipMalloc((void **)&buf.p, bytes);
  if (e != hipSuccess) return e;
  CLeaf *d_lv = (CLeaf *)(buf.p + o_lv);
  double **d_dst = (double **)(buf.p + o_dst);
  int *d_kt = (int *)(buf.p + o_kt), *d_st = (int *)(buf.p + o_st);
  std::vector<int> batch;
  std::vector<CLeaf> lv;
  std::vector<int> kt, st;
  std::vector<double *> dst;
  size_t first = 0;
  for (size_t last : ends) {
    batch.clear();
    lv.clear();
    int n[3] = {0, 0, 0};
    size_t o_b = 0, o_v = 0;
    for (int c = 0; c < 3; ++c)
      for (size_t q = first; q < last; ++q) {
        CLeaf L = d->lv[ids[q]];
        if (aca_class(L) != c) continue;
        L.cap = cap_of(L);
        L.base = (double *)(buf.p + o_b);
        L.pa = (double *)(buf.p + o_pa) + o_v;
        L.msk = (int *)(buf.p + o_msk) + o_v;
        o_b += bytes_of(L);
        o_v += (size_t)L.ndl + L.ndt;
        batch.push_back(ids[q]);
        lv.push_back(L);
        ++n[c];
      }
    first = last;
    const size_t nb = batch.size();
    kt.resize(nb);
    st.resize(nb);
    dst.assign(nb, nullptr);
    if ((e = hipMemcpy(d_lv, lv.data(), sizeof(CLeaf) * nb, hipMemcpyHostToDevice)) != hipSuccess)
      return e;
    if (host_norms)
      launch_aca_class<64, false, true>((int)nb, d_lv, g, p, d_kt, d_st);
    else if (cent)
      launch_aca<true>(n, d_lv, g, p, d_kt, d_st);
    else
      launch_aca<false>(n, d_lv, g, p, d_kt, d_st);
    if ((e = hipGetLastError()) != hipSuccess ||
        (e = hipMemcpy(kt.data(), d_kt, sizeof(int) * nb, hipMemcpyDeviceToHost)) != hipSuccess ||
        (e = hipMemcpy(st.data(), d_st, sizeof(int) * nb, hipMemcpyDeviceToHost)) != hipSuccess)
      return e;
    size_t pool = 0;
    for (size_t q = 0; q < nb; ++q)
      if (st[q] == kAcaOk) pool += ((size_t)lv[q].ndl + lv[q].ndt) * (size_t)kt[q];
    double *d_pool = nullptr;
    if ((e = dalloc(d, (void **)&d_pool, sizeof(double) * pool)) != hipSuccess) return e;
    size_t o = 0;
    for (size_t q = 0; q < nb; ++q) {
      if (st[q] != kAcaOk) {
        (st[q] == kAcaNear ? near : again).push_back(batch[q]);
        continue;
      }
      CLeaf &L = d->lv[batch[q]];
      dst[q] = L.base = d_pool + o;
      L.cap = d->kt[batch[q]] = kt[q];
      o += ((size_t)L.ndl + L.ndt) * (size_t)kt[q];
    }
    if ((e = hipMemcpy(d_dst, dst.data(), sizeof(double *) * nb, hipMemcpyHostToDevice)) !=
        hipSuccess)
      return e;
    // threads per block by its class, as for ACA+
    const int threads[3] = {1024, 256, 64}, parts[3] = {8, 1, 1};
    for (int c = 0, at = 0; c < 3; at += n[c++])
      if (n[c] > 0)
        hipLaunchKernelGGL(k_pack, dim3((unsigned)n[c], parts[c]), dim3(threads[c]), 0, nullptr,
                           d_lv + at, d_kt + at, d_dst + at);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipDeviceSynchronize();
}

}  // namespace

extern "C" {

int hmv_construct(int nnode, const double *nodes, int nface, const int *faces, const double *cent,
                  const double *area, const int *lod, int nlf, const void *specs, int stride,
                  const hmv_construct_params *cp, hmv_dleaves *out) {
  if (!out || !nodes || !faces || !cent || !area || !lod || !specs || !cp || nnode <= 0 ||
      nface <= 0 || nlf < 0 || stride < (int)sizeof(hmv::RefLeaf) ||
      (cp->kernel != kKernelPpohbem && cp->kernel != kKernelCentroid) || cp->kmax < 1 ||
      cp->kmin < 0) {
    hmv::set_error("hmv_construct: invalid argument");
    return HMV_ERR_ARG;
  }
  *out = nullptr;
  for (int64_t i = 0; i < 3 * (int64_t)nface; ++i)
    if (faces[i] < 0 || faces[i] >= nnode) {
      hmv::set_error("hmv_construct: face references a missing node");
      return HMV_ERR_ARG;
    }
  for (int i = 0; i < nface; ++i)
    if (lod[i] < 1 || lod[i] > nface) {
      hmv::set_error("hmv_construct: lod out of range");
      return HMV_ERR_ARG;
    }
  std::unique_ptr<hmv_dleaves_s> d(new hmv_dleaves_s());
  d->nd = nface;
  d->nlf = nlf;
  d->lv.resize(nlf);
  d->kt.assign(nlf, 0);
  std::vector<int> lr_ids;
  std::vector<CLeaf> dense;
  std::vector<int> dense_ids;
  size_t pool = 0;
  for (int i = 0; i < nlf; ++i) {
    const auto *r = reinterpret_cast<const hmv::RefLeaf *>(static_cast<const char *>(specs) +
                                                          (size_t)stride * i);
    CLeaf &L = d->lv[i];
    L = CLeaf{};
    L.ltmtx = r->ltmtx;
    L.nstrtl = r->nstrtl;
    L.ndl = r->ndl;
    L.nstrtt = r->nstrtt;
    L.ndt = r->ndt;
    if ((L.ltmtx != 1 && L.ltmtx != 2) || L.ndl <= 0 || L.ndt <= 0 || L.nstrtl < 1 ||
        L.nstrtt < 1 || (int64_t)L.nstrtl - 1 + L.ndl > nface ||
        (int64_t)L.nstrtt - 1 + L.ndt > nface) {
      hmv::set_error("hmv_construct: leaf " + std::to_string(i + 1) + " outside the matrix");
      return HMV_ERR_ARG;
    }
    if (L.ltmtx == 1) {
      lr_ids.push_back(i);
    } else {
      pool += (size_t)L.ndl * L.ndt;
      dense_ids.push_back(i);
    }
  }
  // device copies for the fill: geometry, then the dense leaf list
  hipError_t e;
  struct Buf {  // freed on every exit
    char *p = nullptr;
    ~Buf() { (void)hipFree(p); }
  } geo;
  const size_t o_area = sizeof(double) * 3 * (size_t)nface,
               o_nodes = o_area + sizeof(double) * (size_t)nface,
               o_dense = o_nodes + sizeof(double) * 3 * (size_t)nnode,
               o_faces = o_dense + sizeof(CLeaf) * dense_ids.size(),
               o_lod = o_faces + sizeof(int) * 3 * (size_t)nface,
               geo_bytes = o_lod + sizeof(int) * (size_t)nface;
  double *d_pool = nullptr;
  if ((e = dalloc(d.get(), (void **)&d_pool, sizeof(double) * pool)) != hipSuccess ||
      (e = hipMalloc((void **)&geo.p, geo_bytes)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_construct: device memory");
  auto t0 = std::chrono::steady_clock::now();
  dense.reserve(dense_ids.size());
  {
    size_t po = 0;
    for (int i : dense_ids) {
      CLeaf &L = d->lv[i];
      L.base = d_pool + po;
      po += (size_t)L.ndl * L.ndt;
      dense.push_back(L);
    }
  }
  auto up = [&](size_t at, const void *src, size_t bytes) {
    if (e == hipSuccess && bytes > 0) e = hipMemcpy(geo.p + at, src, bytes, hipMemcpyHostToDevice);
  };
  up(0, cent, sizeof(double) * 3 * (size_t)nface);
  up(o_area, area, sizeof(double) * (size_t)nface);
  up(o_nodes, nodes, sizeof(double) * 3 * (size_t)nnode);
  up(o_dense, dense.data(), sizeof(CLeaf) * dense.size());
  up(o_faces, faces, sizeof(int) * 3 * (size_t)nface);
  up(o_lod, lod, sizeof(int) * (size_t)nface);
  if (e != hipSuccess) return hmv::hip_fail(e, "hmv_construct: upload");
  Geo g{(double *)geo.p,          (double *)(geo.p + o_area), (double *)(geo.p + o_nodes),
        (int *)(geo.p + o_faces), (int *)(geo.p + o_lod),     cp->kernel};
  AcaParams ap{cp->aca_eps, cp->aca_eps_factor, cp->kmax, cp->kmin};
  // dense leaves
  if (!dense.empty()) {
    hipLaunchKernelGGL(k_dense, dim3((unsigned)dense.size()), dim3(kT), 0, nullptr,
                       (const CLeaf *)(geo.p + o_dense), g);
    if ((e = hipGetLastError()) != hipSuccess)
      return hmv::hip_fail(e, "hmv_construct: dense fill");
  }
  // low-rank leaves, largest first; then the ones that needed more columns, and
  // the ones that hang on the order of a sum
  std::sort(lr_ids.begin(), lr_ids.end(), [&](int a, int b) {
    const int64_t sa = (int64_t)d->lv[a].ndl + d->lv[a].ndt, sb = (int64_t)d->lv[b].ndl + d->lv[b].ndt;
    return sa != sb ? sa > sb : a < b;
  });
  std::vector<int> again, failed, near, none;
  if ((e = run_aca(d.get(), lr_ids, g, ap, first_columns(cp->aca_eps), false, again, near)) !=
          hipSuccess ||
      (e = run_aca(d.get(), again, g, ap, INT_MAX, false, failed, near)) != hipSuccess ||
      (e = run_aca(d.get(), near, g, ap, INT_MAX, true, failed, none)) != hipSuccess ||
      (e = hipDeviceSynchronize()) != hipSuccess)  // the dense fill, if nothing followed it
    return hmv::hip_fail(e, "hmv_construct: ACA+");
  if (!failed.empty()) {
    hmv::set_error("hmv_construct: ACA+ of leaf " + std::to_string(failed[0] + 1) +
                   " exceeded its rank bound");
    return HMV_ERR_STATE;
  }
  auto t1 = std::chrono::steady_clock::now();
  d->seconds = std::chrono::duration<double>(t1 - t0).count();
  // leaf records with device pointers (a2 = a1 + a1size, as the reference)
  d->rec.resize(nlf);
  for (int i = 0; i < nlf; ++i) {
    const CLeaf &L = d->lv[i];
    hmv::RefLeaf &r = d->rec[i];
    std::memset(&r, 0, sizeof(r));
    r.ltmtx = L.ltmtx;
    r.nstrtl = L.nstrtl;
    r.ndl = L.ndl;
    r.nstrtt = L.nstrtt;
    r.ndt = L.ndt;
    r.a1 = L.base;
    if (L.ltmtx == 1) {
      r.kt = d->kt[i];
      r.a1size = (long long)sizeof(double) * L.ndt * L.cap;
      r.a2 = L.base + (size_t)L.ndt * L.cap;
    } else {
      r.kt = 0;
      r.a1size = (long long)sizeof(double) * L.ndl * L.ndt;
      r.a2 = nullptr;
    }
  }
  *out = d.release();
  return HMV_OK;
}

int hmv_dleaves_info(hmv_dleaves d, int *nlf, int *kt, double *seconds) {
  if (!d) {
    hmv::set_error("hmv_dleaves_info: null handle");
    return HMV_ERR_ARG;
  }
  if (nlf) *nlf = d->nlf;
  if (kt) std::copy(d->kt.begin(), d->kt.end(), kt);
  if (seconds) *seconds = d->seconds;
  return HMV_OK;
}

int hmv_dleaves_download(hmv_dleaves d, int leaf, double *a1) {
  if (!d || leaf < 0 || leaf >= d->nlf || !a1) {
    hmv::set_error("hmv_dleaves_download: invalid argument");
    return HMV_ERR_ARG;
  }
  const CLeaf &L = d->lv[leaf];
  hipError_t e;
  if (L.ltmtx == 2) {
    e = hipMemcpy(a1, L.base, sizeof(double) * L.ndl * L.ndt, hipMemcpyDeviceToHost);
  } else {
    const int k = d->kt[leaf];
    e = hipMemcpy(a1, L.base, sizeof(double) * L.ndt * k, hipMemcpyDeviceToHost);
    if (e == hipSuccess)
      e = hipMemcpy(a1 + (size_t)L.ndt * k, L.base + (size_t)L.ndt * L.cap,
                    sizeof(double) * L.ndl * k, hipMemcpyDeviceToHost);
  }
  if (e != hipSuccess) return hmv::hip_fail(e, "hmv_dleaves_download");
  return HMV_OK;
}

int hmv_arena_build_dleaves(hmv_dleaves d, int precision, const hmv_tuning *tuning,
                            hmv_arena *out) {
  if (!d || !out) {
    hmv::set_error("hmv_arena_build_dleaves: null argument");
    return HMV_ERR_ARG;
  }
  return hmv::build_from_device_leaves(d->nd, d->nlf, d->rec.data(), (int)sizeof(hmv::RefLeaf),
                                       precision, tuning, out);
}

int hmv_dleaves_free(hmv_dleaves d) {
  delete d;
  return HMV_OK;
}

}  // extern "C"
