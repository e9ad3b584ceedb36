// hmv_gcr.hip -- GCR(m) on the H-matvec engine, all vectors and scalars on
// the device.
//
// Restates HACApK_gcrm_lfmtx (m_HACApK_solve.f90:506-571) step for step:
//   r = b - A u;  p_1 = r;  ap_1 = A p_1
//   step in (slot ik = (in-1) mod m):
//     alpha = (ap_ik, r) / (ap_ik, ap_ik);  capap_ik = (ap_ik, ap_ik)
//     u += alpha p_ik;  r -= alpha ap_ik;  stop on ||r||/||b|| < eps
//     ar = A r;  new slot ikn = in mod m:  p_ikn = r, ap_ikn = ar, then for
//     il = 1..ik:  beta_il = -(ap_il, ar) / capap_il;
//                  p_ikn += beta_il p_il;  ap_ikn += beta_il ap_il
// When ikn = 1 (in a multiple of m) slot 1 is among 1..ik and was just
// overwritten, so its beta is -(ar, ar)/capap_1 and it scales the new
// direction by (1 + beta_1), as in the reference.  All betas use the
// unmodified ar, so one pass computes them and one fused pass applies them.
// The host feeds the iterations (hmv_feed.h); a device flag set on
// convergence turns those launched after it into no-ops.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <vector>

#include "hmv.h"
#include "hmv_engine.h"
#include "hmv_feed.h"

namespace {

constexpr int kT = 256;
constexpr int kMaxB = kSolveMaxBlocks;
constexpr int kMaxM = HMV_GCR_MAX_M;
constexpr int kMaxBetaB = 128;  // blocks of a beta dot
static_assert(kT == 8 * kMaxM, "8 threads sum the partials of a slot's beta");

struct GcrState {
  double alpha, bnorm, rnorm, eps;
  double capap[kMaxM];
  int step;  // completed steps (the reference's in)
  int ik;    // slot of the current direction (0-based)
  int ikn;   // slot of the next direction (0-based)
  int m, maxit, done, status;
  int ticks;  // iterations ended, with those that found the solve stopped
};

__device__ inline double blk_sum(double v, double *sh) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return r;
}

// part[2*blk + {0,1}]: (a,b), (c,d) partials
__global__ __launch_bounds__(kT) void g_dots2(int n, const double *__restrict__ a,
                                              const double *__restrict__ b,
                                              const double *__restrict__ c,
                                              const double *__restrict__ d,
                                              double *__restrict__ part) {
  __shared__ double sh[4];
  double s0 = 0.0, s1 = 0.0;
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
    s0 = __builtin_fma(a[i], b[i], s0);
    s1 = __builtin_fma(c[i], d[i], s1);
  }
  const double r0 = blk_sum(s0, sh), r1 = blk_sum(s1, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r0;
    part[2 * blockIdx.x + 1] = r1;
  }
}

// (ap_ik, r), (ap_ik, ap_ik) for the slot ik = st->ikn of the first step
// (at setup; g_update_dir produces them for the later steps)
__global__ __launch_bounds__(kT) void g_dots_alpha(int n, const double *__restrict__ ap,
                                                   const double *__restrict__ r,
                                                   double *__restrict__ part, const GcrState *st) {
  if (st->done) return;
  __shared__ double sh[4];
  const double *q = ap + (size_t)st->ikn * n;  // the slot of this step
  double s0 = 0.0, s1 = 0.0;
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
    s0 = __builtin_fma(q[i], r[i], s0);
    s1 = __builtin_fma(q[i], q[i], s1);
  }
  const double r0 = blk_sum(s0, sh), r1 = blk_sum(s1, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r0;
    part[2 * blockIdx.x + 1] = r1;
  }
}

// alpha = (ap_ik, r) / (ap_ik, ap_ik) from the nb partial pairs of
// g_dots_alpha (every block forms it alike; block 0 records it, the slot
// and capap_ik, and flags a breakdown), then u += alpha p_ik;
// r -= alpha ap_ik;  (r, r) partials into rpart (apart is still being read
// by other blocks).
__global__ __launch_bounds__(kT) void g_update_ur(int n, int nb, const double *__restrict__ p,
                                                  const double *__restrict__ ap,
                                                  double *__restrict__ u, double *__restrict__ r,
                                                  const double *__restrict__ apart,
                                                  double *__restrict__ rpart, GcrState *st) {
  __shared__ double sh[4];
  const int done = st->done, ik = st->ikn;  // the slot of this step
  int i = blockIdx.x * kT + threadIdx.x;
  const int i0 = min(i, n - 1);
  double uv = u[i0], rv = r[i0];
  double s0 = 0.0, s1 = 0.0;
  for (int b = threadIdx.x; b < nb; b += kT) {
    s0 += apart[2 * b];
    s1 += apart[2 * b + 1];
  }
  hmv::together(done | ik, uv, rv, s0, s1, 0.0, 0.0, 0.0);
  if (done) return;
  const double *pk = p + (size_t)ik * n, *q = ap + (size_t)ik * n;
  // the first elements are under way while the partials are summed
  double pv = pk[i0], qv = q[i0];
  const double d0 = blk_sum(s0, sh), d1 = blk_sum(s1, sh);
  const double alpha = d0 / d1;
  const bool bad = d1 == 0.0 || !isfinite(alpha);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->ik = ik;
    st->capap[ik] = d1;
    st->alpha = alpha;
    if (bad) {
      st->status = isfinite(d1) ? HMV_SOLVE_BREAKDOWN : HMV_SOLVE_NONFINITE;
      st->done = 1;
    }
  }
  if (bad) return;
  double s2 = 0.0;
  while (i < n) {
    const double ri = rv - alpha * qv;
    u[i] = uv + alpha * pv;
    r[i] = ri;
    s2 = __builtin_fma(ri, ri, s2);
    i += gridDim.x * kT;
    if (i < n) {
      uv = u[i];
      pv = pk[i];
      rv = r[i];
      qv = q[i];
    }
  }
  const double r0 = blk_sum(s2, sh);
  if (threadIdx.x == 0) rpart[blockIdx.x] = r0;
}

// partials of (v_il, ar) for il = 0..ik, v_il = ar for the slot just
// overwritten (il == ikn), else ap_il:  part[blk * kMaxM + il].  Block row
// blockIdx.y covers the kGroup slots from kGroup*blockIdx.y, so ar is read
// once per group.
constexpr int kGroup = 4;
__global__ __launch_bounds__(kT) void g_dots_beta(int n, const double *__restrict__ ap,
                                                  const double *__restrict__ ar,
                                                  double *__restrict__ part, const GcrState *st) {
  const int done = st->done, ik = st->ik, ikn = st->ikn, l0 = blockIdx.y * kGroup;
  int i = blockIdx.x * kT + threadIdx.x;
  double a = ar[min(i, n - 1)];
  hmv::together(done | ik | ikn, a, 0.0, 0.0);
  if (done || l0 > ik) return;
  __shared__ double sh[4];
  const double *v[kGroup];
#pragma unroll
  for (int j = 0; j < kGroup; ++j) {
    const int l = min(l0 + j, ik);
    v[j] = l == ikn ? ar : ap + (size_t)l * n;
  }
  double s[kGroup] = {0.0, 0.0, 0.0, 0.0};
  while (i < n) {
    double x[kGroup];
#pragma unroll
    for (int j = 0; j < kGroup; ++j) x[j] = v[j][i];
    const double ai = a;
    i += gridDim.x * kT;
    if (i < n) a = ar[i];
#pragma unroll
    for (int j = 0; j < kGroup; ++j) s[j] = __builtin_fma(x[j], ai, s[j]);
  }
#pragma unroll
  for (int j = 0; j < kGroup; ++j) {
    const double r0 = blk_sum(s[j], sh);
    if (threadIdx.x == 0 && l0 + j <= ik) part[(size_t)blockIdx.x * kMaxM + l0 + j] = r0;
  }
}

// stage 0: setup (d0 = (r,r), d1 = (b,b) from nb partial pairs); 2: ||r||
// (nb partials), step, stop
__device__ inline void g_publish(HmvSolveHost *h, const GcrState *st) {
  if (st->done) {
    h->step = st->step;
    h->status = st->status;
    h->rnorm = st->rnorm;
    h->bnorm = st->bnorm;
  }
  hmv::publish(h, st->ticks, st->done);
}

__global__ __launch_bounds__(kT) void g_final(int nb, const double *__restrict__ part,
                                              GcrState *st, int stage, double *__restrict__ hist,
                                              HmvSolveHost *h) {
  __shared__ double sh[4];
  double s0 = 0.0, s1 = 0.0;
  if (stage == 0) {
    for (int b = threadIdx.x; b < nb; b += kT) {
      s0 += part[2 * b];
      s1 += part[2 * b + 1];
    }
  } else {
    for (int b = threadIdx.x; b < nb; b += kT) s0 += part[b];
  }
  const int done = st->done, step = st->step, m = st->m, maxit = st->maxit, ticks = st->ticks;
  const double bnorm = st->bnorm, eps = st->eps;
  hmv::together(done | step | m | maxit | ticks, s0, bnorm, eps);
  if (done && stage != 0) {
    if (threadIdx.x == 0) {
      st->ticks = ticks + 1;
      g_publish(h, st);
    }
    return;
  }
  const double d0 = blk_sum(s0, sh), d1 = blk_sum(s1, sh);
  if (threadIdx.x != 0) return;
  if (stage == 0) {
    st->rnorm = sqrt(d0);
    st->bnorm = sqrt(d1);
    st->step = 0;
    st->ik = 0;
    st->ikn = 0;
    st->done = 0;
    st->status = HMV_SOLVE_MAXITER;
    if (hist) hist[0] = st->rnorm / st->bnorm;
    if (!isfinite(st->rnorm) || !isfinite(st->bnorm) || st->bnorm == 0.0) {
      st->status = HMV_SOLVE_NONFINITE;
      st->done = 1;
    } else if (st->rnorm / st->bnorm < st->eps) {
      st->status = HMV_SOLVE_CONVERGED;
      st->done = 1;
    } else if (st->maxit <= 0) {
      st->done = 1;
    }
    st->ticks = 0;
  } else {
    const double rnorm = sqrt(d0), rel = rnorm / bnorm;
    st->step = step + 1;
    st->rnorm = rnorm;
    st->ikn = (step + 1) % m;
    st->ticks = ticks + 1;
    if (hist) hist[step + 1] = rel;
    int status = -1;
    if (!isfinite(rnorm))
      status = HMV_SOLVE_NONFINITE;
    else if (rel < eps)
      status = HMV_SOLVE_CONVERGED;
    else if (step + 1 >= maxit)
      status = HMV_SOLVE_MAXITER;
    if (status < 0) {
      hmv::publish(h, ticks + 1, 0);
      return;
    }
    st->status = status;
    st->done = 1;
  }
  g_publish(h, st);
}

// beta_l = -(v_l, ar) / capap_l for the slots l <= ik, from the nbb partials
// of g_dots_beta: every block sums them alike, 8 threads a slot, into sb.  A
// launch of its own for this took 4.7 us of a step at 82k unknowns.
__device__ inline void form_betas(int nbb, const double *__restrict__ bpart,
                                  const double *__restrict__ capap, int ik, double *sb) {
  const int l = threadIdx.x >> 3, sub = threadIdx.x & 7;
  const double cap = capap[min(l, ik)];
  double v = 0.0;
  for (int b = sub; b < nbb; b += 8) v += bpart[(size_t)b * kMaxM + min(l, ik)];
  for (int off = 4; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if (sub == 0) sb[l] = -v / cap;
  __syncthreads();
}

// p_ikn = c0 r + sum_{il <= ik, il != ikn} beta_il p_il;  ap_ikn likewise
// with ar;  c0 = 1 + beta_ikn when ikn <= ik (slot 1 at a restart), else 1
// ... and the next step's alpha partials (ap_ikn, r), (ap_ikn, ap_ikn) into
// part[2*blk + {0,1}], in g_dots_alpha's order (same grid, same per-thread
// sequence), so that the step needs no separate dot pass.
// An element's slots are loaded kDir at a time, a group ahead of its sums and
// the first one ahead of the betas: one at a time leaves a chain of up to m
// loads per thread, which is what the pass takes at a few elements each.
constexpr int kDir = 8;
__global__ __launch_bounds__(kT) void g_update_dir(int n, int nbb, const double *__restrict__ r,
                                                   const double *__restrict__ ar,
                                                   double *__restrict__ p, double *__restrict__ ap,
                                                   const double *__restrict__ bpart,
                                                   double *__restrict__ part, const GcrState *st) {
  __shared__ double sh[4], sb[kMaxM];
  const int done = st->done, ik = st->ik, ikn = st->ikn;
  int i = blockIdx.x * kT + threadIdx.x;
  const int i0 = min(i, n - 1);
  double rv = r[i0], av0 = ar[i0];
  hmv::together(done | ik | ikn, rv, av0, 0.0);
  if (done) return;
  double pl[kDir], al[kDir];
  auto load = [&](int l0, int at) {
#pragma unroll
    for (int j = 0; j < kDir; ++j) {
      pl[j] = p[(size_t)min(l0 + j, ik) * n + at];
      al[j] = ap[(size_t)min(l0 + j, ik) * n + at];
    }
  };
  load(0, i0);
  form_betas(nbb, bpart, st->capap, ik, sb);
  const double c0 = ikn <= ik ? 1.0 + sb[ikn] : 1.0;
  double *pn = p + (size_t)ikn * n, *apn = ap + (size_t)ikn * n;
  double s0 = 0.0, s1 = 0.0;
  const int stride = gridDim.x * kT;
  while (i < n) {
    const double ri = rv;
    double pv = c0 * ri, av = c0 * av0;
    for (int l0 = 0; l0 <= ik; l0 += kDir) {
      double pc[kDir], ac[kDir];
#pragma unroll
      for (int j = 0; j < kDir; ++j) {
        pc[j] = pl[j];
        ac[j] = al[j];
      }
      if (l0 + kDir <= ik) {
        load(l0 + kDir, i);
      } else if (i + stride < n) {
        rv = r[i + stride];
        av0 = ar[i + stride];
        load(0, i + stride);
      }
#pragma unroll
      for (int j = 0; j < kDir; ++j) {
        if (l0 + j > ik || l0 + j == ikn) continue;
        const double bl = sb[l0 + j];
        pv = __builtin_fma(bl, pc[j], pv);
        av = __builtin_fma(bl, ac[j], av);
      }
    }
    pn[i] = pv;
    apn[i] = av;
    s0 = __builtin_fma(av, ri, s0);
    s1 = __builtin_fma(av, av, s1);
    i += stride;
  }
  const double r0 = blk_sum(s0, sh), r1 = blk_sum(s1, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r0;
    part[2 * blockIdx.x + 1] = r1;
  }
}

// r = b - ar (r = b when ar is null: a zero initial guess);  p_1 = r; the
// state's parameters (st may be null)
__global__ __launch_bounds__(kT) void g_init(int n, const double *__restrict__ b,
                                             const double *__restrict__ ar,
                                             double *__restrict__ r, double *__restrict__ p,
                                             GcrState *st, double eps, int m, int maxit) {
  if (st && blockIdx.x == 0 && threadIdx.x == 0) {
    st->eps = eps;
    st->m = m;
    st->maxit = maxit;
  }
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
    const double ri = ar ? b[i] - ar[i] : b[i];
    r[i] = ri;
    p[i] = ri;
  }
}

int grid_of(int n) {
  return std::max(1, std::min((n + kT - 1) / kT, kMaxB));
}

// Blocks of a beta dot: 4 elements per thread, and few enough that every
// block of g_update_dir can sum the partials of all of them.
int beta_grid(int n) { return std::max(1, std::min((n + 4 * kT - 1) / (4 * kT), kMaxBetaB)); }

}  // namespace

// GCR workspace, kept with the arena between calls.
struct HmvGcrWork {
  int m = 0;
  size_t hist_cap = 0;
  hipStream_t s = nullptr;
  double *r = nullptr, *ar = nullptr, *p = nullptr, *ap = nullptr, *part = nullptr, *bpart = nullptr,
         *hist = nullptr;
  GcrState *st = nullptr;
  double *ir_r = nullptr, *ir_d = nullptr;  // refinement: outer residual, correction
  ~HmvGcrWork() {
    if (s) (void)hipStreamDestroy(s);
    for (double *q : {r, ar, p, ap, part, bpart, hist, ir_r, ir_d}) (void)hipFree(q);
    (void)hipFree(st);
  }
};

namespace hmv {
void free_gcr_work(hmv_arena_s *a) {
  delete a->gcr;
  a->gcr = nullptr;
}
}  // namespace hmv

namespace {

using GcrWork = HmvGcrWork;

// The arena's GCR workspace for m directions and maxit steps.
int gcr_work(hmv_arena_s *a, int m, int maxit, GcrWork *&out) {
  GcrWork *w = a->gcr;
  if (w && (w->m != m || w->hist_cap < (size_t)maxit + 1)) {
    hmv::free_gcr_work(a);
    w = nullptr;
  }
  if (!w) {
    w = new GcrWork();
    a->gcr = w;
    const int n = a->nd, g = grid_of(n);
    const size_t nb = sizeof(double) * (size_t)n;
    w->m = m;
    w->hist_cap = (size_t)maxit + 1;
    hipError_t e;
    if ((e = hipStreamCreateWithFlags(&w->s, hipStreamNonBlocking)) != hipSuccess ||
        (e = hipMalloc(&w->r, nb)) != hipSuccess || (e = hipMalloc(&w->ar, nb)) != hipSuccess ||
        (e = hipMalloc(&w->p, nb * m)) != hipSuccess || (e = hipMalloc(&w->ap, nb * m)) != hipSuccess ||
        (e = hipMalloc(&w->part, sizeof(double) * 3 * (size_t)g)) != hipSuccess ||
        (e = hipMalloc(&w->bpart, sizeof(double) * (size_t)beta_grid(n) * kMaxM)) != hipSuccess ||
        (e = hipMalloc(&w->hist, sizeof(double) * w->hist_cap)) != hipSuccess ||
        (e = hipMalloc(&w->st, sizeof(GcrState))) != hipSuccess) {
      hmv::free_gcr_work(a);
      return hmv::hip_fail(e, "hmv_gcrm: workspace");
    }
  }
  out = w;
  return HMV_OK;
}

hipError_t gcr_iteration(hmv_arena_s *a, GcrWork &w, int n, int m, double *u, HmvSolveHost *h) {
  const int g = grid_of(n), gb = beta_grid(n);
  const int *skip = &w.st->done;
  // (r, r) partials at [2g, 3g) of the partials, apart from the alpha pairs
  // at [0, 2g) that g_update_ur reads while writing them
  double *rpart = w.part + 2 * (size_t)g;
  // the alpha partials of this step come from the previous step's
  // g_update_dir (or, for the first step, from the setup's g_dots_alpha)
  hipLaunchKernelGGL(g_update_ur, dim3(g), dim3(kT), 0, w.s, n, g, w.p, w.ap, u, w.r,
                     (const double *)w.part, rpart, w.st);
  hipLaunchKernelGGL(g_final, dim3(1), dim3(kT), 0, w.s, g, (const double *)rpart, w.st, 2, w.hist,
                     h);
  hipError_t e = hmv::enqueue_apply(a, w.r, w.ar, 0.0, skip, w.s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(g_dots_beta, dim3(gb, (m + kGroup - 1) / kGroup), dim3(kT), 0, w.s, n, w.ap,
                     w.ar, w.bpart, (const GcrState *)w.st);
  hipLaunchKernelGGL(g_update_dir, dim3(g), dim3(kT), 0, w.s, n, gb, w.r, w.ar, w.p, w.ap,
                     (const double *)w.bpart, w.part, (const GcrState *)w.st);
  return hipGetLastError();
}

}  // namespace

namespace {
int gcrm_run(hmv_arena a, const double *b, double *u, double eps, int maxit, int m,
             double *hist, hmv_solve_info *info, bool true_res,
             bool zero_guess = false);
}

extern "C" int hmv_gcrm(hmv_arena a, const double *b, double *u, double eps, int maxit, int m,
                        int /*check_every*/, double *hist, hmv_solve_info *info) {
  return gcrm_run(a, b, u, eps, maxit, m, hist, info, true);
}

namespace {
// true_res: recompute ||b - A u|| / ||b|| at the end (one more product).
// zero_guess: u is known to be zero, so r = b without the product A u.
int gcrm_run(hmv_arena a, const double *b, double *u, double eps, int maxit, int m,
             double *hist, hmv_solve_info *info, bool true_res,
             bool zero_guess) {
  if (!a || !b || !u || maxit < 0 || m < 1 || m > kMaxM) {
    hmv::set_error("hmv_gcrm: invalid argument (1 <= m <= 32)");
    return HMV_ERR_ARG;
  }
  const int n = a->nd, g = grid_of(n);
  GcrWork *wp = nullptr;
  int rc = gcr_work(a, m, maxit, wp);
  if (rc) return rc;
  GcrWork &w = *wp;
  hipError_t e;
  HmvSolveHost *h = nullptr;
  if ((e = hmv::solve_host(a, w.s, h)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_gcrm: workspace");
  auto t0 = std::chrono::steady_clock::now();
  if (!zero_guess && (e = hmv::enqueue_apply(a, u, w.ar, 0.0, nullptr, w.s)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_gcrm: setup");
  hipLaunchKernelGGL(g_init, dim3(g), dim3(kT), 0, w.s, n, b, zero_guess ? nullptr : w.ar, w.r,
                     w.p, w.st, eps, m, maxit);
  hipLaunchKernelGGL(g_dots2, dim3(g), dim3(kT), 0, w.s, n, w.r, w.r, b, b, w.part);
  hipLaunchKernelGGL(g_final, dim3(1), dim3(kT), 0, w.s, g, w.part, w.st, 0, w.hist, h);
  // ap_1 = A p_1 (skipped when already converged) and the first step's
  // alpha partials
  if ((e = hmv::enqueue_apply(a, w.p, w.ap, 0.0, &w.st->done, w.s)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_gcrm: setup");
  hipLaunchKernelGGL(g_dots_alpha, dim3(g), dim3(kT), 0, w.s, n, w.ap, w.r, w.part,
                     (const GcrState *)w.st);
  if ((e = hipGetLastError()) != hipSuccess) return hmv::hip_fail(e, "hmv_gcrm: setup");
  int launched = 0;
  e = hmv::feed(h, w.s, launched, maxit,
                [&] { return gcr_iteration(a, w, n, m, u, h); });
  // the refinement goes on on the same stream; a caller's u is complete here
  if (e == hipSuccess && (true_res || !hmv::stopped(h))) e = hipStreamSynchronize(w.s);
  if (e != hipSuccess) return hmv::hip_fail(e, "hmv_gcrm: iterations");
  auto t1 = std::chrono::steady_clock::now();
  if (hist) {
    std::fill(hist, hist + maxit + 1, NAN);
    if ((e = hipMemcpy(hist, w.hist, sizeof(double) * ((size_t)h->step + 1),
                       hipMemcpyDeviceToHost)) != hipSuccess)
      return hmv::hip_fail(e, "hmv_gcrm: history");
  }
  // true residual ||b - A u|| / ||b||
  double tr = NAN;
  if (true_res) {
    if ((e = hmv::enqueue_apply(a, u, w.ar, 0.0, nullptr, w.s)) != hipSuccess)
      return hmv::hip_fail(e, "hmv_gcrm: true residual");
    hipLaunchKernelGGL(g_init, dim3(g), dim3(kT), 0, w.s, n, b, w.ar, w.r, w.p,
                       (GcrState *)nullptr, 0.0, 0, 0);
    hipLaunchKernelGGL(g_dots2, dim3(g), dim3(kT), 0, w.s, n, w.r, w.r, b, b, h->part);
    if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(w.s)) != hipSuccess)
      return hmv::hip_fail(e, "hmv_gcrm: true residual");
    double rr = 0.0, bb = 0.0;
    for (int i = 0; i < g; ++i) {
      rr += h->part[2 * i];
      bb += h->part[2 * i + 1];
    }
    tr = std::sqrt(rr) / std::sqrt(bb);
  }
  if (info) {
    info->nstp = h->step;
    info->status = h->status;
    info->relres = h->rnorm / h->bnorm;
    info->true_relres = tr;
    info->seconds = std::chrono::duration<double>(t1 - t0).count();
    info->outer = 0;
    info->inner_total = h->step;
  }
  return HMV_OK;
}
}  // namespace

namespace {

// r = b - v
__global__ __launch_bounds__(kT) void g_residual(int n, const double *__restrict__ b,
                                                 const double *__restrict__ v,
                                                 double *__restrict__ r) {
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) r[i] = b[i] - v[i];
}

// u += d;  d = 0
__global__ __launch_bounds__(kT) void g_add_clear(int n, double *__restrict__ u,
                                                  double *__restrict__ d) {
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
    u[i] = u[i] + d[i];
    d[i] = 0.0;
  }
}

// r = b - A u and ||r|| / ||b|| (A: the arena a) on stream s; the partial
// dots go to h
int residual(hmv_arena_s *a, hipStream_t s, HmvSolveHost *h, const double *b, const double *u,
             double *v, double *r, double *rel) {
  const int n = a->nd, g = grid_of(n);
  hipError_t e;
  if ((e = hmv::enqueue_apply(a, u, v, 0.0, nullptr, s)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_gcr_ir: residual");
  hipLaunchKernelGGL(g_residual, dim3(g), dim3(kT), 0, s, n, b, v, r);
  hipLaunchKernelGGL(g_dots2, dim3(g), dim3(kT), 0, s, n, r, r, b, b, h->part);
  if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(s)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_gcr_ir: residual");
  double rr = 0.0, bb = 0.0;
  for (int i = 0; i < g; ++i) {
    rr += h->part[2 * i];
    bb += h->part[2 * i + 1];
  }
  *rel = std::sqrt(rr) / std::sqrt(bb);
  return HMV_OK;
}

}  // namespace

extern "C" int hmv_gcr_ir(hmv_arena a64, hmv_arena alow, const double *b, double *u, double eps,
                          double inner_eps, int m, int max_outer, int max_inner, int /*check_every*/,
                          double *hist, hmv_solve_info *info) {
  if (!a64 || !alow || !b || !u || a64->nd != alow->nd || m < 1 || m > kMaxM || max_outer < 0 ||
      max_inner < 0) {
    hmv::set_error("hmv_gcr_ir: invalid arguments");
    return HMV_ERR_ARG;
  }
  const int n = a64->nd, g = grid_of(n);
  const size_t nb = sizeof(double) * (size_t)n;
  // everything runs on the stream of the low-precision arena's workspace,
  // whose ar holds A64 u between the inner solves
  GcrWork *wp = nullptr;
  int rc = gcr_work(alow, m, max_inner, wp);
  if (rc) return rc;
  GcrWork &w = *wp;
  HmvSolveHost *h = nullptr;
  hipError_t e;
  if ((!w.ir_r && (e = hipMalloc(&w.ir_r, nb)) != hipSuccess) ||
      (!w.ir_d && (e = hipMalloc(&w.ir_d, nb)) != hipSuccess) ||
      (e = hmv::solve_host(alow, w.s, h)) != hipSuccess ||
      (e = hipMemsetAsync(w.ir_d, 0, nb, w.s)) != hipSuccess)
    return hmv::hip_fail(e, "hmv_gcr_ir: workspace");
  auto t0 = std::chrono::steady_clock::now();
  double rel = 0.0;
  rc = residual(a64, w.s, h, b, u, w.ar, w.ir_r, &rel);
  if (rc) return rc;
  if (hist) hist[0] = rel;
  int outer = 0, inner_total = 0, status = HMV_SOLVE_MAXITER;
  if (!std::isfinite(rel)) status = HMV_SOLVE_NONFINITE;
  while (status == HMV_SOLVE_MAXITER && rel >= eps && outer < max_outer) {
    // solve Alow d = r to inner_eps with GCR(m), d starting at zero
    hmv_solve_info in{};
    rc = gcrm_run(alow, w.ir_r, w.ir_d, inner_eps, max_inner, m, nullptr, &in, false, true);
    if (rc) return rc;
    inner_total += in.nstp;
    if (in.status == HMV_SOLVE_NONFINITE) status = HMV_SOLVE_NONFINITE;
    hipLaunchKernelGGL(g_add_clear, dim3(g), dim3(kT), 0, w.s, n, u, w.ir_d);
    ++outer;
    rc = residual(a64, w.s, h, b, u, w.ar, w.ir_r, &rel);
    if (rc) return rc;
    if (hist) hist[outer] = rel;
    if (!std::isfinite(rel)) status = HMV_SOLVE_NONFINITE;
  }
  if (status == HMV_SOLVE_MAXITER && rel < eps) status = HMV_SOLVE_CONVERGED;
  auto t1 = std::chrono::steady_clock::now();
  if (info) {
    info->nstp = inner_total;
    info->status = status;
    info->relres = rel;
    info->true_relres = rel;
    info->seconds = std::chrono::duration<double>(t1 - t0).count();
    info->outer = outer;
    info->inner_total = inner_total;
  }
  return HMV_OK;
}
