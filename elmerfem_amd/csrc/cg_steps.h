// The Krylov scalars' updates and stopping tests that the launched loops
// (krylov.hip) and the resident loops (resident.hip) both run.
#pragma once
#include "ehip_internal.h"
#include "linalg_kernels.h"
#include "reduce.h"

namespace ehip {

template <typename T>
__device__ __forceinline__ bool solve_done(const KStateT<T> *st) {
  // `done` only changes at the end of an earlier launch, so a plain load is
  // coherent here; it is uniform, so it becomes one scalar load per wave
  // instead of a same-address L2 request from every lane
  return __builtin_amdgcn_readfirstlane(st->done) != 0;
}

// The unscaled relative residual ||b - A x|| / ||b|| from the sum of squares
// of r_s / D on the scaled system (r_s = D0 (b - A x) / beta and D = D0 beta,
// so r_s / D = (b - A x) / beta^2, and likewise b_s / D = b / beta^2).
// Records it and tells whether it meets tol_u; true when the test is off.
template <typename T>
__device__ __forceinline__ bool unscaled_ok(KStateT<T> *st, T sum_u) {
  if (!(st->tol_u > (T)0)) return true;
  const T ru = sqrt(sum_u / st->bb_u);
  st->res_u = ru;
  return ru < st->tol_u;
}

#define EHIP_EPI_MEMBERS(T) \
  Vecs<T> v;                \
  KStateT<T> *st;           \
  T *partials;              \
  int stride;               \
  unsigned *ticket;

// The stopping tests on the recurrence residual after a CG vector step, in
// the order HUTI applies them: converged, diverged, rho = 0, out of
// iterations, and (mixed form) a reliable update due.
struct CgCheck {
  int done, info, rec_conv;
};
template <typename T>
__device__ __forceinline__ CgCheck cg_check(T res, T rz, int it, const KStateT<T> *st) {
  if (res < st->tol) return {1, 0, 1};
  if (!(res == res) || (st->divtol > (T)0 && res > st->divtol)) return {1, 3, 0};
  if (rz == (T)0) return {1, 20, 0};
  if (it >= st->maxit) return {1, 2, 0};
  if (res < st->ru) return {1, 0, 2};  // reliable update due
  return {0, 0, 0};
}
template <typename T>
__device__ __forceinline__ void cg_apply(const CgCheck &c, KStateT<T> *st) {
  if (c.rec_conv) st->rec_conv = c.rec_conv;
  if (c.info) st->info = c.info;
  if (c.done) st->done = 1;
}

template <typename T>
struct FinCgFast2 {
  static constexpr int NV = 2;
  KStateT<T> *st;
  T *partials;
  int stride;
  double *hist;
  __device__ void finish(T (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const T rho_old = st->rho;
    st->rho_new = rho_old;  // kept for a residual replacement, which recomputes beta
    st->rho = tot[0];
    st->beta = tot[0] / rho_old;
    st->rr = tot[1];
    const T res = sqrt(tot[1]) / st->rhsnorm;
    st->res = res;
    const int it = st->iter + 1;  // iterations done
    st->iter = it;
    if (hist && it - 1 < st->maxit) hist[it - 1] = (double)res;
    cg_apply(cg_check(res, tot[0], it, st), st);
  }
};

template <typename T>
struct EpiCgResidual {
  static constexpr int NV = 2;
  EHIP_EPI_MEMBERS(T)
  double *hist;
  const T *rn_part;  // Kda's partials of rho_new = r.z
  int rn_g;
  T beta;
  const T *du;  // the scaling's D, or null when the unscaled test is off
  // rho_new summed from Kda's partials by every workgroup in the same order
  // (workgroup 0 records it for the finalize), in place of a finalize launch
  __device__ void init() {
    T rn[1];
    block_reduce_all<T, 1>(rn_part, 0, rn_g, rn);
    if (blockIdx.x == 0 && threadIdx.x == 0) st->rho_new = rn[0];
    beta = rn[0] / st->rho;
  }
  struct Pre { T b, z, p, d; };
  __device__ Pre load(int i) const { return Pre{v.b[i], v.z[i], v.p[i], du ? du[i] : (T)1}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[2]) {
    const T ti = s - pr.b;
    acc[0] += ti * ti;
    const T ui = ti / pr.d;
    acc[1] += ui * ui;
    v.p[i] = pr.z + beta * pr.p;
  }
  __device__ void finish(T (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const T res = sqrt(tot[0]) / st->rhsnorm;
    st->res = res;
    const int it = st->iter;  // HUTI iter_count, 1-based
    if (hist && it - 1 < st->maxit) hist[it - 1] = (double)res;
    if (res < st->tol && unscaled_ok(st, tot[1])) {
      st->info = 1;
      st->done = 1;
      return;
    }
    st->rho = st->rho_new;
    st->iter = it + 1;
    if (it + 1 > st->maxit) {
      st->info = 2;
      st->done = 1;
    } else if (st->rho_new == (T)0) {
      st->info = 20;
      st->done = 1;
    }
  }
};

template <typename T>
struct FinSnorm {
  static constexpr int NV = 1;
  KStateT<T> *st;
  T *partials;
  int stride;
  __device__ void finish(T (&tot)[1]) {
    if (threadIdx.x != 0) return;
    const T sn = sqrt(tot[0]);
    st->snorm = sn;
    if (sn < (T)1.17549435E-38f) {  // HUTI_EPSILON (huti_fdefs.h)
      st->snorm_exit = 1;
      st->info = 36;
    }
  }
};

template <typename T>
struct FinBiXr {
  static constexpr int NV = 2;
  KStateT<T> *st;
  T *partials;
  int stride;
  int fast;
  double *hist;
  __device__ void finish(T (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const T alpha = st->alpha, omega = st->omega;
    st->rho_new = tot[0];
    st->rr = tot[1];
    if (fast) {
      const T res = sqrt(tot[1]) / st->rhsnorm;
      st->res = res;
      const int it = st->iter;
      if (hist && it - 1 < st->maxit) hist[it - 1] = (double)res;
      if (res < st->tol) {
        st->rec_conv = 1;
        st->done = 1;
        return;
      }
      if (!(res == res) || (st->divtol > (T)0 && res > st->divtol)) {
        st->info = 3;
        st->done = 1;
        return;
      }
      if (omega == (T)0) {
        st->info = 37;
        st->done = 1;
        return;
      }
      st->iter = it + 1;
      if (it + 1 > st->maxit) {
        st->info = 2;
        st->done = 1;
      } else if (tot[0] == (T)0) {
        st->info = 35;
        st->done = 1;
      } else {
        st->beta = (tot[0] * alpha) / (st->rho * omega);
        st->rho = tot[0];
      }
    }
  }
};

template <typename T>
struct EpiBiResidual {
  static constexpr int NV = 2;
  EHIP_EPI_MEMBERS(T)
  double *hist;
  T beta, omega;
  const T *du;  // the scaling's D, or null when the unscaled test is off
  __device__ void init() {
    omega = st->omega;
    beta = (st->rho_new * st->alpha) / (st->rho * omega);
  }
  struct Pre { T b, r, p, v, dg, d; };
  __device__ Pre load(int i) const { return Pre{v.b[i], v.r[i], v.p[i], v.v[i], v.dg[i], du ? du[i] : (T)1}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[2]) {
    const T ti = s - pr.b;
    acc[0] += ti * ti;
    const T ui = ti / pr.d;
    acc[1] += ui * ui;
    const T pi = pr.r + beta * (pr.p - omega * pr.v);
    v.p[i] = pi;
    v.t1v[i] = pi / pr.dg;
  }
  __device__ void finish(T (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const T res = sqrt(tot[0]) / st->rhsnorm;
    st->res = res;
    const int it = st->iter;
    if (hist && it - 1 < st->maxit) hist[it - 1] = (double)res;
    if (res < st->tol && unscaled_ok(st, tot[1])) {
      st->info = 1;
      st->done = 1;
      return;
    }
    if (st->omega == (T)0) {
      st->info = 37;
      st->done = 1;
      return;
    }
    st->iter = it + 1;
    if (it + 1 > st->maxit) {
      st->info = 2;
      st->done = 1;
    } else if (st->rho_new == (T)0) {
      st->info = 35;
      st->done = 1;
    } else {
      st->rho = st->rho_new;
    }
  }
};

}  // namespace ehip
