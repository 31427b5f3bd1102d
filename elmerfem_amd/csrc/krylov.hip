// Scaling, Dirichlet rows and the Krylov solvers of libehip.
//
// The solve follows SolveLinearSystem's iterative branch
// (fem/src/SolverUtils.src:7151-7525): zero-RHS exit, ScaleLinearSystem
// (:6470-6640), x = 1e-8 when x = 0 (IterSolve.src:358), HUTI CG
// (hutiter/src/huti_cg.src:73-244) or BiCGStab (huti_bicgstab.src:85-273)
// with the TRESID_SCALED_BYB stop test, BackScaleLinearSystem (:6754-6866)
// and ComputeNorm (:4887-5006).
//
// Every reduction is two launches on the solve's stream: the producing
// kernel publishes one partial per workgroup with plain stores and a
// one-workgroup finalize sums them in a fixed order (run-to-run
// deterministic) and updates the Krylov scalars.  Every kernel reads the
// device-side `done` flag first and returns when the solve has ended, so the
// host enqueues blocks of iterations and polls the scalars only every
// `check_every` iterations.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "cg_steps.h"
#include "ehip_internal.h"
#include "launch.h"
#include "linalg_kernels.h"
#include "spmv_core.h"

namespace ehip {

thread_local GraphRec *tl_graph_rec = nullptr;
thread_local hipError_t tl_launch_err = hipSuccess;
thread_local bool tl_shared_device = false;

// Whether the mixed form's FP32 CG runs its folded two-launch steps
// (EHIP_CG_FOLD=0 turns them off: three launches per iteration).  Read at
// every block of iterations, so a process can compare the two.
static bool cg_fold_enabled() {
  const char *f = std::getenv("EHIP_CG_FOLD");
  return !(f && f[0] == '0');
}

bool graphs_enabled() {
  static const bool on = [] {
    const char *g = std::getenv("EHIP_GRAPHS");
    if (g && *g) return g[0] != '0';
    return std::getenv("ROCPROF_OUTPUT_PATH") == nullptr;
  }();
  return on;
}

// ---------------------------------------------------------------- scaling

// D_i = 1/sqrt(|a_ii|); a zero diagonal falls back to the row's absolute
// sum (ScaleLinearSystem, SolverUtils.src:6520-6550).
__global__ void k_diag_scale(int n, const int *__restrict__ rows, const int *__restrict__ diag,
                             const double *__restrict__ vals, double *__restrict__ D) {
  const double tiny = DBL_MIN;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double d = vals[diag[i]];
    if (fabs(d) <= tiny) {
      double s = 0.0;
      for (int j = rows[i]; j < rows[i + 1]; ++j) s += fabs(vals[j]);
      d = s;
    }
    D[i] = fabs(d) > tiny ? 1.0 / sqrt(fabs(d)) : 1.0;
  }
}

struct ScaleValues {
  double *vals;
  const int *cols;
  const double *D;
  float *v32;  // optional FP32 copy of the scaled values
  __device__ void operator()(int r, int j) {
    double v = vals[j] * (D[r] * D[cols[j]]);
    vals[j] = v;
    if (v32) v32[j] = (float)v;
  }
};

struct BackscaleValues {
  double *vals;
  const int *cols;
  const double *D;
  __device__ void operator()(int r, int j) { vals[j] = vals[j] / (D[r] * D[cols[j]]); }
};

// b *= D and the sum of squares of the scaled b (ScaleLinearSystem's bnorm)
__global__ __launch_bounds__(kVecBlock) void k_scale_rhs(int n, double *__restrict__ b,
                                                         const double *__restrict__ D, double *partials,
                                                         unsigned *ticket, double *out) {
  double acc[1] = {0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double v = b[i] * D[i];
    b[i] = v;
    acc[0] += v * v;
  }
  (void)ticket;
  (void)out;
  block_publish<double, 1>(acc, partials, gridDim.x);
}

// one workgroup: *out = sum of g partials
__global__ __launch_bounds__(256) void k_fin_sum(const double *partials, int g, double *out) {
  double tot[1];
  block_reduce_all<double, 1>(partials, g, g, tot);
  if (threadIdx.x == 0) *out = tot[0];
}

// D *= bnorm; b /= bnorm; x /= D
__global__ void k_scale_rhs2(int n, double *b, double *D, double *x, double bnorm) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double d = D[i] * bnorm;
    D[i] = d;
    b[i] = b[i] / bnorm;
    if (x) x[i] = x[i] / d;
  }
}

// the same with ||b|| from device memory (sqrt of the finalized sum of squares)
__global__ void k_scale_rhs2_dev(int n, double *b, double *D, double *x, const double *ss, double *bnorm_out) {
  const double bnorm = sqrt(*ss);
  if (blockIdx.x == 0 && threadIdx.x == 0) *bnorm_out = bnorm;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double d = D[i] * bnorm;
    D[i] = d;
    b[i] = b[i] / bnorm;
    if (x) x[i] = x[i] / d;
  }
}

// BackScaleLinearSystem vector part: x *= D; D /= bnorm; b = b / D * bnorm
__global__ void k_backscale_vec_dev(int n, double *b, double *D, double *x, const double *bn) {
  const double bnorm = *bn;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    if (x) x[i] = x[i] * D[i];
    double d = D[i] / bnorm;
    D[i] = d;
    b[i] = b[i] / d * bnorm;
  }
}

__global__ void k_backscale_vec(int n, double *b, double *D, double *x, double bnorm) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    if (x) x[i] = x[i] * D[i];
    double d = D[i] / bnorm;
    D[i] = d;
    b[i] = b[i] / d * bnorm;
  }
}

int scale_system(ehip_system *s, double *b, bool rhs_scaling, double *x, double *bnorm_out, bool make_f32,
                 double *bnorm_dev) {
  const int n = s->n;
  int rc;
  if ((rc = ensure_state(s))) return rc;
  if (make_f32 && !s->vals32)
    if ((rc = dmalloc(s, (void **)&s->vals32, sizeof(float) * s->nnz))) return rc;
  hipLaunchKernelGGL(k_diag_scale, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, s->rows, s->diag,
                     s->vals, s->dscale);
  ScaleValues f{s->vals, s->cols, s->dscale, make_f32 ? s->vals32 : nullptr};
  hipLaunchKernelGGL(k_nonzeros<ScaleValues>, dim3(s->plan64.grid), dim3(256), 0, s->stream, s->rows,
                     s->plan64.chunk_row, s->plan64.nchunks, f);
  touch_vals(s, true, make_f32);
  double bnorm = 1.0;
  if (b) {
    double *dsum = reinterpret_cast<double *>(&s->st->ts);
    const int g = vec_grid(n);
    hipLaunchKernelGGL(k_scale_rhs, dim3(g), dim3(kVecBlock), 0, s->stream, n, b, s->dscale, s->partials,
                       &s->st->ticket[0], dsum);
    hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(256), 0, s->stream, s->partials, g, dsum);
    if (rhs_scaling && bnorm_dev) {
      // ||b|| stays on the device: nothing waits here
      hipLaunchKernelGGL(k_scale_rhs2_dev, dim3(g), dim3(kVecBlock), 0, s->stream, n, b, s->dscale, x,
                         (const double *)dsum, bnorm_dev);
      EHIP_HIP_TRY(hipGetLastError());
      return EHIP_OK;
    }
    if (rhs_scaling) {
      double ss = 0;
      EHIP_HIP_TRY(hipMemcpyAsync(&ss, dsum, sizeof(double), hipMemcpyDeviceToHost, s->stream));
      EHIP_HIP_TRY(hipStreamSynchronize(s->stream));
      bnorm = sqrt(ss);
    }
    hipLaunchKernelGGL(k_scale_rhs2, dim3(g), dim3(kVecBlock), 0, s->stream, n, b, s->dscale, x, bnorm);
  }
  if (bnorm_out) *bnorm_out = bnorm;
  EHIP_HIP_TRY(hipGetLastError());
  return EHIP_OK;
}

int backscale_system(ehip_system *s, double *b, double *x, double rhs_scale, const double *rhs_scale_dev) {
  const int n = s->n;
  if (b && rhs_scale_dev)
    hipLaunchKernelGGL(k_backscale_vec_dev, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, b, s->dscale, x,
                       rhs_scale_dev);
  else if (b)
    hipLaunchKernelGGL(k_backscale_vec, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, b, s->dscale, x,
                       rhs_scale);
  BackscaleValues f{s->vals, s->cols, s->dscale};
  hipLaunchKernelGGL(k_nonzeros<BackscaleValues>, dim3(s->plan64.grid), dim3(256), 0, s->stream, s->rows,
                     s->plan64.chunk_row, s->plan64.nchunks, f);
  touch_vals(s, true, false);
  EHIP_HIP_TRY(hipGetLastError());
  return EHIP_OK;
}

// ---------------------------------------------------------------- Dirichlet

// DefaultDirichletBCs on a scaled system without RHS scaling: every value is
// taken through v*(D_i D_j) and back through /(D_i D_j) like the reference's
// scale / back-scale round trip; Dirichlet rows become a unit diagonal in
// the scaled system (ZeroRow + SetMatrixElement, SolverUtils.src:2632-2657)
// or, in symmetric mode, their columns are eliminated into b
// (CRS_SetSymmDirichlet, CRSMatrix.src:674-735).
struct DirichletValues {
  double *vals;
  const int *cols;
  const double *D;
  const signed char *isbc;
  int symmetric;
  __device__ void operator()(int r, int j) {
    const int c = cols[j];
    double v = vals[j] * (D[r] * D[c]);
    if (isbc[r]) v = (c == r) ? 1.0 : 0.0;
    else if (symmetric && isbc[c]) v = 0.0;
    vals[j] = v / (D[r] * D[c]);
  }
};

__global__ void k_fill1(int n, double *d) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) d[i] = 1.0;
}

// rhs: b*D, Dirichlet b = val/D, symmetric elimination b -= a_ij val_j/D_j,
// then b/D.  `vals` are still the unscaled, pre-Dirichlet values here.
__global__ void k_dirichlet_rhs(int n, const int *__restrict__ rows, const int *__restrict__ cols,
                                const double *__restrict__ vals, double *b, const double *__restrict__ D,
                                const signed char *__restrict__ isbc, const double *__restrict__ bcval,
                                int symmetric) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double bi = b[i] * D[i];
    if (isbc[i]) {
      bi = bcval[i] / D[i];
    } else if (symmetric) {
      for (int j = rows[i]; j < rows[i + 1]; ++j) {
        const int c = cols[j];
        if (isbc[c]) bi = bi - vals[j] * (D[i] * D[c]) * (bcval[c] / D[c]);
      }
    }
    b[i] = bi / D[i];
  }
}

}  // namespace ehip

using namespace ehip;

extern "C" int ehip_dirichlet(ehip_system *s, int nbc, const int *bc_rows, const double *bc_vals, int symmetric,
                              int scaling) {
  if (!s || nbc < 0 || (nbc > 0 && !bc_rows)) return EHIP_EARG;
  const int n = s->n;
  int rc;
  // the rows and values go to the device once; a call with the same ones
  // (re-assembly with new coefficients on the same mesh) only enqueues kernels
  const bool same = s->bc_flag && (int)s->h_bc_rows.size() == nbc &&
                    std::equal(bc_rows, bc_rows + nbc, s->h_bc_rows.begin()) &&
                    (bc_vals ? (s->h_bc_vals.size() == (size_t)nbc &&
                                std::equal(bc_vals, bc_vals + nbc, s->h_bc_vals.begin()))
                             : s->h_bc_vals.empty());
  if (!same) {
    std::vector<signed char> flag(n, 0);
    std::vector<double> val(n, 0.0);
    for (int k = 0; k < nbc; ++k) {
      int r = bc_rows[k];
      if (r < 1 || r > n) {
        set_error("ehip_dirichlet: row %d out of range", r);
        return EHIP_EARG;
      }
      flag[r - 1] = 1;
      val[r - 1] = bc_vals ? bc_vals[k] : 0.0;
    }
    if (!s->bc_flag && (rc = dmalloc(s, (void **)&s->bc_flag, n))) return rc;
    if (!s->bc_val && (rc = dmalloc(s, (void **)&s->bc_val, sizeof(double) * n))) return rc;
    EHIP_HIP_TRY(hipMemcpyAsync(s->bc_flag, flag.data(), n, hipMemcpyHostToDevice, s->stream));
    EHIP_HIP_TRY(hipMemcpyAsync(s->bc_val, val.data(), sizeof(double) * n, hipMemcpyHostToDevice, s->stream));
    EHIP_HIP_TRY(hipStreamSynchronize(s->stream));  // the host vectors go out of scope
    s->h_bc_rows.assign(bc_rows, bc_rows + nbc);
    if (bc_vals) s->h_bc_vals.assign(bc_vals, bc_vals + nbc);
    else s->h_bc_vals.clear();
  }
  if ((rc = ensure_state(s))) return rc;
  double *D = s->dscale;
  if (scaling) {
    hipLaunchKernelGGL(k_diag_scale, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, s->rows, s->diag,
                       s->vals, D);
  } else {
    hipLaunchKernelGGL(k_fill1, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, D);
  }
  hipLaunchKernelGGL(k_dirichlet_rhs, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, s->rows, s->cols,
                     s->vals, s->rhs, D, s->bc_flag, s->bc_val, symmetric);
  DirichletValues f{s->vals, s->cols, D, s->bc_flag, symmetric};
  hipLaunchKernelGGL(k_nonzeros<DirichletValues>, dim3(s->plan64.grid), dim3(256), 0, s->stream, s->rows,
                     s->plan64.chunk_row, s->plan64.nchunks, f);
  touch_vals(s, true, false);
  EHIP_HIP_TRY(hipGetLastError());
  return EHIP_OK;
}

namespace ehip {

// ================================================================ Krylov kernels

// r = b - A x ; z = r/dg ; partials r.z, r.r, b.b  (start of every solve)
template <typename T>
struct EpiInit {
  static constexpr int NV = 3;
  EHIP_EPI_MEMBERS(T)
  __device__ void init() {}
  struct Pre { T b, dg; };
  __device__ Pre load(int i) const { return Pre{v.b[i], v.dg[i]}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[3]) {
    const T bi = pr.b;
    const T ri = bi - s;
    v.r[i] = ri;
    const T zi = ri / pr.dg;
    v.z[i] = zi;
    acc[0] += ri * zi;
    acc[1] += ri * ri;
    acc[2] += bi * bi;
  }
  __device__ void finish(T (&tot)[3]) {
    if (threadIdx.x == 0) {
      st->rhsnorm = sqrt(tot[2]);
      st->rho = tot[0];
      st->rr = tot[1];
      st->res = sqrt(tot[1]) / st->rhsnorm;
      st->beta = (T)0;
    }
  }
};

template <typename T, int BS, int NB, class CS, class Epi>
__global__ __launch_bounds__(BS) void k_spmv_epi(const int *__restrict__ rows, const int *__restrict__ c32,
                                                 const unsigned short *__restrict__ c16,
                                                 const int *__restrict__ segb, const T *__restrict__ vals,
                                                 const T *__restrict__ xin, const int *__restrict__ chunk_row,
                                                 int nchunks, Epi epi, const KStateT<T> *st) {
  if (st && solve_done(st)) return;
  const CS cols(c32, c16, segb);
  spmv_stream_body<T, T, BS, NB>(rows, cols, vals, xin, chunk_row, nchunks, epi);
}

// ---- fast CG, 1 SpMV per iteration
// step 1: q = A z + beta q ; p = z + beta p ; partial p.q -> alpha
template <typename T>
struct EpiCgFast1 {
  static constexpr int NV = 1;
  EHIP_EPI_MEMBERS(T)
  T beta;
  __device__ void init() { beta = st->beta; }
  struct Pre { T q, z, p; };
  __device__ Pre load(int i) const { return Pre{v.q[i], v.z[i], v.p[i]}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[1]) {
    const T qi = s + beta * pr.q;
    const T pi = pr.z + beta * pr.p;
    v.q[i] = qi;
    v.p[i] = pi;
    acc[0] += pi * qi;
  }
  __device__ void finish(T (&tot)[1]) {
    if (threadIdx.x == 0) {
      st->pq = tot[0];
      st->alpha = st->rho / tot[0];
    }
  }
};

// One tile of the CG vector step: x, p, r, q and the Jacobi diagonal of
// kVI elements per lane.
template <typename T>
struct CgTile {
  T x[kVI], p[kVI], r[kVI], q[kVI], d[kVI];
  __device__ __forceinline__ void load(const Vecs<T> &v, int n, int base) {
#pragma unroll
    for (int k = 0; k < kVI; ++k) {
      const int i = base + k * kVecBlock + threadIdx.x;
      if (i < n) { x[k] = v.x[i]; p[k] = v.p[i]; r[k] = v.r[i]; q[k] = v.q[i]; d[k] = v.dg[i]; }
    }
  }
  // x += alpha p ; r -= alpha q ; z = r/dg ; acc += r.z (and r.r when NA = 2)
  template <int NA>
  __device__ __forceinline__ void step(const Vecs<T> &v, int n, int base, T alpha, T (&acc)[NA]) const {
#pragma unroll
    for (int k = 0; k < kVI; ++k) {
      const int i = base + k * kVecBlock + threadIdx.x;
      if (i < n) {
        v.x[i] = x[k] + alpha * p[k];
        const T ri = r[k] - alpha * q[k];
        v.r[i] = ri;
        const T zi = ri / d[k];
        v.z[i] = zi;
        acc[0] += ri * zi;
        if constexpr (NA > 1) acc[1] += ri * ri;
      }
    }
  }
};

// alpha = rho / p.q, summed from the SpMV step's partials by every workgroup
// in the same fixed order (so all agree bit for bit; workgroup 0 records it)
// -- this replaces a one-workgroup finalize launch.  The first tile's loads
// do not depend on alpha and go out before the reduction, so the two
// latencies overlap.  Then x += alpha p ; r -= alpha q ; z = r/dg with the
// partials of r.z (and r.r when NA = 2).
template <typename T, int NA, bool Fold = false>
__device__ __forceinline__ void cg_vector_step(int n, const Vecs<T> &v, KStateT<T> *st, const T *pq_part, int pq_g,
                                               T *partials) {
  const int stride = gridDim.x * kVecBlock * kVI;
  int base = blockIdx.x * kVecBlock * kVI;
  CgTile<T> cur, nxt;
  cur.load(v, n, base);
  T pq[1];
  block_reduce_all<T, 1>(pq_part, 0, pq_g, pq);
  // folded steps: rho was summed by the SpMV step before (rho_next); this
  // launch makes it current and counts the iteration
  const T alpha = (Fold ? st->rho_next : st->rho) / pq[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->pq = pq[0];
    st->alpha = alpha;
    if constexpr (Fold) {
      st->rho = st->rho_next;
      st->iter = st->iter + 1;
      st->fresh = 0;
    }
  }
  T acc[NA];
#pragma unroll
  for (int k = 0; k < NA; ++k) acc[k] = (T)0;
  while (base < n) {
    const int nb = base + stride;
    if (nb < n) nxt.load(v, n, nb);
    cur.template step<NA>(v, n, base, alpha, acc);
    cur = nxt;
    base = nb;
  }
  block_publish<T, NA>(acc, partials, gridDim.x);
}

// step 2 of the one-SpMV CG: partials r.z, r.r
template <typename T, bool Fold = false>
__global__ __launch_bounds__(kVecBlock) void k_cg_fast2(int n, Vecs<T> v, KStateT<T> *st, const T *pq_part,
                                                        int pq_g, T *partials) {
  if (solve_done(st)) return;
  if constexpr (Fold) {
    // the SpMV step before stopped the sequence (its state is already final)
    if (__builtin_amdgcn_readfirstlane(st->stop_pending)) {
      if (blockIdx.x == 0 && threadIdx.x == 0) st->done = 1;
      return;
    }
  }
  cg_vector_step<T, 2, Fold>(n, v, st, pq_part, pq_g, partials);
}

// ---- folded FP32 CG steps (the inner sequence of the mixed form): two
// launches per iteration instead of three.  The SpMV step opens by summing
// the previous vector step's partials (r.z, r.r) itself -- every workgroup,
// in the one-workgroup finalize's order, so every workgroup gets that
// finalize's bits -- and runs its stopping tests.  Fields of the state each
// launch reads and writes, so that no workgroup reads a field that another
// workgroup of the same launch writes:
//   SpMV step   reads  done, fresh, rho, iter, maxit, tol, divtol, ru, rhsnorm (beta when fresh);
//               writes rho_next, rr, res, and on a stop rho_new, rho, beta, info, rec_conv,
//               stop_pending.  A stop is decided by every workgroup alike from the same
//               sums (neither the decision nor the work it skips reads rho or beta).
//   vector step reads  done, stop_pending, rho_next; writes pq, alpha, rho = rho_next,
//               iter + 1, fresh = 0 -- or, after a stop, only done = 1.
// The SpMV step must not write `done` itself: every kernel tests it on entry
// once per wavefront, and a wavefront that started after the write would
// return while the other wavefronts of its workgroup, which started before
// it, go on into the workgroup barriers of the reduction without it and sum
// unwritten LDS slots -- a wrong beta for their rows.  (It happened only when
// the workgroups of one launch were spread out in time, i.e. with other
// solves running on the device.)  stop_pending is written by one launch and
// read, alike by every wavefront, by the next.
// A block of folded iterations ends with FinCgFold, the finalize of the last
// vector step, which leaves rho and beta current (fresh = 1) as the start
// and a residual replacement do.  The state then matches the unfolded
// sequence's after the same number of iterations, bit for bit.
constexpr int kFoldPer = 4;
static_assert(kFusedCap <= kFoldPer * 256, "vector-step partials must fit the SpMV prologue's loads");

template <typename T>
struct EpiCgFold {
  static constexpr int NV = 1;
  EHIP_EPI_MEMBERS(T)
  const T *rz_part;  // the vector step's partials: r.z at [0, rz_g), r.r at [rz_g, 2 rz_g)
  int rz_g;
  T beta;
  bool skip;
  __device__ void init() {
    skip = false;
    if (st->fresh) {
      beta = st->beta;
      if (blockIdx.x == 0 && threadIdx.x == 0) st->rho_next = st->rho;
      return;
    }
    T tot[2];
    block_reduce_few<T, 2, kFoldPer>(rz_part, rz_g, rz_g, tot);
    const T rho_old = st->rho;
    const T res = sqrt(tot[1]) / st->rhsnorm;
    const CgCheck c = cg_check(res, tot[0], st->iter, st);
    beta = tot[0] / rho_old;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (c.done) {
      skip = true;
      if (lead) {
        st->rho_new = rho_old;
        st->rho = tot[0];
        st->beta = beta;
        st->rr = tot[1];
        st->res = res;
        if (c.rec_conv) st->rec_conv = c.rec_conv;
        if (c.info) st->info = c.info;
        st->stop_pending = 1;
      }
      return;
    }
    if (lead) {
      st->rho_next = tot[0];
      st->rr = tot[1];
      st->res = res;
    }
  }
  struct Pre { T q, z, p; };
  __device__ Pre load(int i) const { return Pre{v.q[i], v.z[i], v.p[i]}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[1]) {
    const T qi = s + beta * pr.q;
    const T pi = pr.z + beta * pr.p;
    v.q[i] = qi;
    v.p[i] = pi;
    acc[0] += pi * qi;
  }
  __device__ void finish(T (&)[1]) {}
};

// end of a block of folded iterations: FinCgFast2's scalar update and tests
// for the last vector step (whose launch already counted the iteration),
// leaving rho and beta current
template <typename T>
struct FinCgFold {
  static constexpr int NV = 2;
  KStateT<T> *st;
  T *partials;
  int stride;
  __device__ void finish(T (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const T rho_old = st->rho;
    st->rho_new = rho_old;
    st->rho = tot[0];
    st->beta = tot[0] / rho_old;
    st->rr = tot[1];
    const T res = sqrt(tot[1]) / st->rhsnorm;
    st->res = res;
    cg_apply(cg_check(res, tot[0], st->iter, st), st);
    st->fresh = 1;
  }
};

// The one-workgroup finalize: sums the producing launch's partials in a
// fixed order and runs its scalar update.  Skipped, like its producer, once
// the solve is done.
template <typename T, class Fin>
__global__ __launch_bounds__(256) void k_fin(Fin f, int g, const KStateT<T> *check) {
  if (check && solve_done(check)) return;
  T tot[Fin::NV];
  block_reduce_all<T, Fin::NV>(f.partials, f.stride, g, tot);
  f.finish(tot);
}

// true residual t = b - A x ; restart r = t, z = t/dg ; partials t.t, t.z
// and (unscaled test on) (t/D).(t/D)
template <typename T>
struct EpiTrue {
  static constexpr int NV = 3;
  EHIP_EPI_MEMBERS(T)
  const T *du;  // the scaling's D, or null when the unscaled test is off
  __device__ void init() {}
  struct Pre { T b, dg, d; };
  __device__ Pre load(int i) const { return Pre{v.b[i], v.dg[i], du ? du[i] : (T)1}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[3]) {
    const T ti = pr.b - s;
    v.r[i] = ti;
    const T zi = ti / pr.dg;
    v.z[i] = zi;
    acc[0] += ti * ti;
    acc[1] += ti * zi;
    const T ui = ti / pr.d;
    acc[2] += ui * ui;
  }
  __device__ void finish(T (&tot)[3]) {
    if (threadIdx.x == 0) {
      const T rt = sqrt(tot[0]) / st->rhsnorm;
      const T rho_prev = st->rho_new;  // r.z before the last step (FinCgFast2)
      st->res_true = rt;
      st->rho = tot[1];
      st->rr = tot[0];
      st->beta = (T)0;
      st->done = 0;
      st->rec_conv = 0;
      const bool ok_s = rt < st->tol;
      if (ok_s && unscaled_ok(st, tot[2])) {
        st->info = 1;
        st->done = 1;
      } else if (st->iter >= st->maxit) {
        st->info = 2;
        st->done = 1;
      } else if (ok_s) {
        // the scaled test holds but the unscaled residual still misses tol_u:
        // the recurrence test is tightened by the observed ratio of the two
        // and the CG direction continues through this residual replacement
        st->tol = rt * (st->tol_u / st->res_u);
        st->beta = rho_prev != (T)0 ? tot[1] / rho_prev : (T)0;
      }
    }
  }
};

// ---- faithful CG in huti_cg.src order; per iteration k:
//   Kc : q = A p ; alpha = rho / (p.q)
//   Kda: x += alpha p ; r -= alpha q ; z = r/dg ; rho_new = r.z
//   Ke : t = A x - b ; residual ||t||/||b|| ; p = z + (rho_new/rho) p
template <typename T>
struct EpiCgQ {
  static constexpr int NV = 1;
  EHIP_EPI_MEMBERS(T)
  __device__ void init() {}
  struct Pre { T p; };
  __device__ Pre load(int i) const { return Pre{v.p[i]}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[1]) {
    v.q[i] = s;
    acc[0] += pr.p * s;
  }
  __device__ void finish(T (&tot)[1]) {
    if (threadIdx.x == 0) {
      st->pq = tot[0];
      st->alpha = st->rho / tot[0];
    }
  }
};

// HUTI order: alpha = rho / p.q from Kc's partials, then the vector step
// with the partials of rho_new = r.z
template <typename T>
__global__ __launch_bounds__(kVecBlock) void k_cg_da(int n, Vecs<T> v, KStateT<T> *st, const T *pq_part,
                                                     int pq_g, T *partials) {
  if (solve_done(st)) return;
  cg_vector_step<T, 1>(n, v, st, pq_part, pq_g, partials);
}

// ---- BiCGStab in huti_bicgstab.src order; per iteration k:
//   B3 : v = A t1v ; alpha = rho / (rtld.v)
//   B45: s = r - alpha v ; t2v = s/dg ; ||s|| (s-norm exit below HUTI_EPSILON)
//   B6 : t = A t2v ; omega = (t.s)/(t.t)
//   B71: x += alpha t1v + omega t2v ; r = s - omega t ; rho_new = rtld.r
//   B82: faithful: residual ||A x - b||/||b|| fused with p = r + beta (p - omega v), t1v = p/dg
//        fast    : residual ||r||/||b|| inside B71, p update as a vector kernel
template <typename T>
struct EpiBiV {
  static constexpr int NV = 1;
  EHIP_EPI_MEMBERS(T)
  __device__ void init() {}
  struct Pre { T rtld; };
  __device__ Pre load(int i) const { return Pre{v.rtld[i]}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[1]) {
    v.v[i] = s;
    acc[0] += pr.rtld * s;
  }
  __device__ void finish(T (&tot)[1]) {
    if (threadIdx.x == 0) st->alpha = st->rho / tot[0];
  }
};

template <typename T>
__global__ __launch_bounds__(kVecBlock) void k_bi_s(int n, Vecs<T> v, KStateT<T> *st, T *partials) {
  if (solve_done(st)) return;
  const T alpha = st->alpha;
  T acc[1] = {(T)0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const T si = v.r[i] - alpha * v.v[i];
    v.sv[i] = si;
    v.t2v[i] = si / v.dg[i];
    acc[0] += si * si;
  }
  block_publish<T, 1>(acc, partials, gridDim.x);
}

template <typename T>
struct EpiBiT {
  static constexpr int NV = 2;
  EHIP_EPI_MEMBERS(T)
  int active;
  __device__ void init() { active = !st->snorm_exit; }
  struct Pre { T sv; };
  __device__ Pre load(int i) const { return Pre{v.sv[i]}; }
  __device__ void row(int i, T s, const Pre &pr, T (&acc)[2]) {
    v.t[i] = s;
    acc[0] += s * pr.sv;
    acc[1] += s * s;
  }
  __device__ void finish(T (&tot)[2]) {
    if (threadIdx.x == 0) {
      st->ts = tot[0];
      st->tt = tot[1];
      st->omega = tot[0] / tot[1];
    }
  }
};

// s-norm exit: x += alpha t1v and finish
template <typename T>
__global__ void k_bi_snorm_exit(int n, Vecs<T> v, KStateT<T> *st) {
  if (solve_done(st) || !st->snorm_exit) return;
  const T alpha = st->alpha;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    v.x[i] = v.x[i] + alpha * v.t1v[i];
}
template <typename T>
__global__ void k_bi_snorm_mark(KStateT<T> *st) {
  if (!st->done && st->snorm_exit) st->done = 1;
}

template <typename T>
__global__ __launch_bounds__(kVecBlock) void k_bi_xr(int n, Vecs<T> v, KStateT<T> *st, T *partials, int fast,
                                                     double *hist) {
  if (solve_done(st)) return;
  const T alpha = st->alpha, omega = st->omega;
  T acc[2] = {(T)0, (T)0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    v.x[i] = v.x[i] + alpha * v.t1v[i] + omega * v.t2v[i];
    const T ri = v.sv[i] - omega * v.t[i];
    v.r[i] = ri;
    acc[0] += v.rtld[i] * ri;
    acc[1] += ri * ri;
  }
  (void)fast;
  (void)hist;
  block_publish<T, 2>(acc, partials, gridDim.x);
}

// fast BiCGStab p update: p = r + beta (p - omega v) ; t1v = p/dg
template <typename T>
__global__ void k_bi_p(int n, Vecs<T> v, KStateT<T> *st) {
  if (solve_done(st)) return;
  const T beta = st->beta, omega = st->omega;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const T pi = v.r[i] + beta * (v.p[i] - omega * v.v[i]);
    v.p[i] = pi;
    v.t1v[i] = pi / v.dg[i];
  }
}

// BiCGStab start: rtld = r ; first p = r (beta = 0, p = v = 0) ; t1v = p/dg ; rho = rtld.r
template <typename T>
__global__ __launch_bounds__(kVecBlock) void k_bi_start(int n, Vecs<T> v, KStateT<T> *st, T *partials) {
  if (solve_done(st)) return;
  T acc[1] = {(T)0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const T ri = v.r[i];
    v.rtld[i] = ri;
    v.p[i] = ri;
    v.v[i] = (T)0;
    v.t1v[i] = ri / v.dg[i];
    acc[0] += ri * ri;
  }
  block_publish<T, 1>(acc, partials, gridDim.x);
}

template <typename T>
struct FinBiStart {
  static constexpr int NV = 1;
  KStateT<T> *st;
  T *partials;
  int stride;
  __device__ void finish(T (&tot)[1]) {
    if (threadIdx.x != 0) return;
    st->rho = tot[0];
    st->omega = (T)1;
    st->alpha = (T)0;
    if (tot[0] == (T)0) {
      st->info = 35;
      st->done = 1;
    }
  }
};

// dg = a_ii, or 1 when |a_ii| <= AEPS or without preconditioning (CRS_DiagPrecondition)
template <typename T>
__global__ void k_make_dg(int n, const int *__restrict__ diag, const double *__restrict__ vals, T *dg, int precond) {
  const double AEPS = 10.0 * DBL_EPSILON;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double d = vals[diag[i]];
    dg[i] = (T)((precond && fabs(d) > AEPS) ? d : 1.0);
  }
}

template <typename T>
__global__ void k_fill(int n, T *x, T val) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) x[i] = val;
}

template <typename T>
__global__ void k_zero2(int n, T *a, T *b) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    a[i] = (T)0;
    b[i] = (T)0;
  }
}

template <typename T>
__global__ void k_init_state(KStateT<T> *st, T tol, int maxit, T divtol, int iter0, T tol_u) {
  st->tol = tol;
  st->tol_u = tol_u;
  st->res_u = (T)-1;
  st->maxit = maxit;
  st->divtol = divtol;
  st->iter = iter0;
  st->info = 0;
  st->done = 0;
  st->snorm_exit = 0;
  st->rec_conv = 0;
  st->beta = (T)0;
  st->rho_new = (T)0;
  st->ru = (T)0;
  st->res_true = (T)-1;
  st->pad0 = 0;
  st->pad1 = 0;
  st->rho_next = (T)0;
  st->fresh = 1;
  st->stop_pending = 0;
}

// ---- mixed precision
// r32 = t/||t|| ; z32 = r32/dg32 ; d32 = 0 ; rho, rr in FP32
__global__ __launch_bounds__(kVecBlock) void k_to32(int n, const double *__restrict__ t, double inv, float *r,
                                                    float *z, float *d, const float *__restrict__ dg,
                                                    KState32 *st, float *partials) {
  float acc[2] = {0.f, 0.f};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float ri = (float)(t[i] * inv);
    r[i] = ri;
    const float zi = ri / dg[i];
    z[i] = zi;
    d[i] = 0.f;
    acc[0] += ri * zi;
    acc[1] += ri * ri;
  }
  (void)st;
  block_publish<float, 2>(acc, partials, gridDim.x);
}

struct FinTo32 {
  static constexpr int NV = 2;
  KState32 *st;
  float *partials;
  int stride;
  __device__ void finish(float (&tot)[2]) {
    if (threadIdx.x != 0) return;
    st->rho = tot[0];
    st->rr = tot[1];
    st->rhsnorm = sqrtf(tot[1]);
    st->beta = 0.f;
    st->iter = 0;
    st->done = 0;
    st->info = 0;
    st->rec_conv = 0;
  }
};

// x64 += scale * d32
__global__ void k_correct(int n, double *x, const float *__restrict__ d, double scale) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    x[i] = x[i] + scale * (double)d[i];
}

// FP64 outer residual: t = b - A x ; partial t.t -> res_true, scale = ||t||
// (and (t/D).(t/D) for the unscaled test)
struct EpiOuter {
  static constexpr int NV = 2;
  double *b, *t;
  KState *st;
  double *partials;
  int stride;
  unsigned *ticket;
  double *hist;
  const double *du;  // the scaling's D, or null when the unscaled test is off
  __device__ void init() {}
  struct Pre { double b, d; };
  __device__ Pre load(int i) const { return Pre{b[i], du ? du[i] : 1.0}; }
  __device__ void row(int i, double s, const Pre &pr, double (&acc)[2]) {
    const double ti = pr.b - s;
    t[i] = ti;
    acc[0] += ti * ti;
    const double ui = ti / pr.d;
    acc[1] += ui * ui;
  }
  __device__ void finish(double (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const double nt = sqrt(tot[0]);
    st->scale = nt;
    const double res = nt / st->rhsnorm;
    st->res_true = res;
    st->res = res;
    const int k = st->pad0;  // outer step
    if (hist && k < st->maxit) hist[k] = res;
    st->pad0 = k + 1;
    if (res < st->tol && unscaled_ok(st, tot[1])) {
      st->info = 1;
      st->done = 1;
    } else if (!(res == res)) {
      st->info = 3;
      st->done = 1;
    }
  }
};

// Residual replacement of the reliable-update mixed CG, on the FP64 matrix:
// t = b - A x64 ; r32 = t ; z32 = r32/dg32 ; x32 = 0 ; partials t.t, r32.z32.
// The caller has folded x32 into x64 (k_correct) first.  The finalize sets
// the FP64 outer residual and restarts the FP32 recurrence from r32 with the
// search direction kept: rho = r32.z32 and beta = rho / (r.z of the step
// before), so the next FP32 step continues the same CG sequence.
struct EpiRU {
  static constexpr int NV = 3;
  const double *b;
  Vecs<float> v;
  KState *st;
  KState32 *st32;
  double *partials;
  int stride;
  unsigned *ticket;
  double *hist;
  double delta;  // next replacement when the FP32 residual has dropped by this factor
  const double *du;  // the scaling's D, or null when the unscaled test is off
  __device__ void init() {}
  struct Pre { double b, d; float dg; };
  __device__ Pre load(int i) const { return Pre{b[i], du ? du[i] : 1.0, v.dg[i]}; }
  __device__ void row(int i, double s, const Pre &pr, double (&acc)[3]) {
    const double t = pr.b - s;
    const float r = (float)t;
    const float z = r / pr.dg;
    v.r[i] = r;
    v.z[i] = z;
    v.x[i] = 0.f;
    acc[0] += t * t;
    acc[1] += (double)(r * z);
    const double u = t / pr.d;
    acc[2] += u * u;
  }
  __device__ void finish(double (&tot)[3]) {
    if (threadIdx.x != 0) return;
    const double res = sqrt(tot[0]) / st->rhsnorm;
    st->res_true = res;
    st->res = res;
    const int k = st->pad0;  // replacement count
    if (hist && k < st->maxit) hist[k] = res;
    st->pad0 = k + 1;
    const float rz = (float)tot[1];
    const float rho_prev = st32->rho_new;
    st32->rho = rz;
    st32->beta = rho_prev != 0.f ? rz / rho_prev : 0.f;
    st32->res = (float)res;
    const bool ok_s = res < st->tol;
    if (ok_s && unscaled_ok(st, tot[2])) {
      st->info = 1;
      st->done = 1;
    } else if (!(res == res)) {
      st->info = 3;
      st->done = 1;
    } else {
      // scaled test met, unscaled not yet: the FP32 sequence's own stop
      // threshold is tightened by the observed ratio of the two residuals
      if (ok_s) st32->tol = fminf(st32->tol, (float)(res * (st->tol_u / st->res_u)));
      st32->ru = (float)(res * delta);
      st32->rec_conv = 0;
      st32->done = 0;
      st32->stop_pending = 0;
      st32->fresh = 1;
    }
  }
};

// rhsnorm = sqrt(rr) in both states (after sumsq into st->rr)
__global__ void k_set_rhsnorm(KState *st, KState32 *st32) {
  const double bn = sqrt(st->rr);
  st->rhsnorm = bn;
  st32->rhsnorm = (float)bn;
}

// sum of squares of b and of b - A x (unscaled report residual)
struct EpiResid {
  static constexpr int NV = 2;
  const double *b;
  double *partials;
  int stride;
  unsigned *ticket;
  double *out;
  __device__ void init() {}
  struct Pre { double b; };
  __device__ Pre load(int i) const { return Pre{b[i]}; }
  __device__ void row(int i, double s, const Pre &pr, double (&acc)[2]) {
    const double t = pr.b - s;
    acc[0] += t * t;
    acc[1] += pr.b * pr.b;
  }
  __device__ void finish(double (&tot)[2]) {
    if (threadIdx.x == 0) {
      out[0] = tot[0];
      out[1] = tot[1];
    }
  }
};

// partials of sum_i (x_i / d_i)^2 (d null: sum_i x_i^2)
__global__ __launch_bounds__(kVecBlock) void k_sumsq(int n, const double *x, const double *d, double *partials,
                                                     unsigned *ticket, double *out) {
  double acc[1] = {0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double u = d ? x[i] / d[i] : x[i];
    acc[0] += u * u;
  }
  (void)ticket;
  (void)out;
  block_publish<double, 1>(acc, partials, gridDim.x);
}

// ================================================================ host drivers

template <typename T, class CS, class Epi>
static void launch_epi_cs(ehip_system *s, const SpmvPlan &p, const T *vals, const T *xin, const Epi &e,
                          const KStateT<T> *st) {
#define EHIP_EPI_CASE(BS, NB)                                                                               \
  if (p.block == BS && p.nb == NB) {                                                                        \
    if (s->prof_start)                                                                                      \
      hipExtLaunchKernelGGL((k_spmv_epi<T, BS, NB, CS, Epi>), dim3(p.grid), dim3(BS), 0, s->stream,         \
                            s->prof_start, s->prof_stop, 0, s->rows, s->cols, s->cols16, s->seg_base, vals,  \
                            xin, p.chunk_row, p.nchunks, e, st);                                             \
    else                                                                                                    \
      launch_k((k_spmv_epi<T, BS, NB, CS, Epi>), dim3(p.grid), dim3(BS), s->stream, s->rows, s->cols,       \
               s->cols16, s->seg_base, vals, xin, p.chunk_row, p.nchunks, e, st);                           \
    return;                                                                                                 \
  }
  EHIP_SPMV_CONFIGS(EHIP_EPI_CASE)
#undef EHIP_EPI_CASE
}

template <typename T, int BS, int U, bool C16, class Epi>
__global__ __launch_bounds__(BS) void k_spmv_epi_sell(const int *__restrict__ rows, int n, const int *__restrict__ rmap,
                                                      const int *__restrict__ c32,
                                                      const unsigned short *__restrict__ c16,
                                                      const int *__restrict__ sbase, const int *__restrict__ off,
                                                      const T *__restrict__ vals, const T *__restrict__ xin,
                                                      int nslice, Epi epi, const KStateT<T> *st) {
  if (st && solve_done(st)) return;
  const SellCols<C16> sc{c32, c16, sbase};
  spmv_sell_body<T, T, BS, U>(rows, n, rmap, sc, off, vals, xin, nslice, epi);
}

template <typename T, int BS, int U, int D, bool NT, class Epi>
__global__ __launch_bounds__(BS) void k_spmv_epi_sho(int n, const int *__restrict__ off, const int *__restrict__ tab,
                                                     const unsigned *__restrict__ mask, const T *__restrict__ vals,
                                                     const T *__restrict__ xin, int nslice, int nt_from,
                                                     Epi epi, const KStateT<T> *st) {
  if (st && solve_done(st)) return;
  spmv_sho_body<T, T, BS, U, D, NT>(n, off, tab, mask, vals, xin, nslice, nt_from, epi);
}

template <int BS, int U, class Epi>
__global__ __launch_bounds__(BS) void k_spmv_epi_sell2(const int *__restrict__ rows, int n, const int *__restrict__ rmap,
                                                       const unsigned short *__restrict__ c16,
                                                       const int *__restrict__ sbase, const int *__restrict__ off2,
                                                       const double *__restrict__ vals, const double *__restrict__ xin,
                                                       int nslice, Epi epi, const KState *st) {
  if (st && solve_done(st)) return;
  spmv_sell2_body<double, BS, U>(rows, n, rmap, c16, sbase, off2, vals, xin, nslice, epi);
}

template <typename T, int BS, int U, int D, class Epi>
__global__ __launch_bounds__(BS) void k_spmv_epi_sellb(const int *__restrict__ rows, int n, const int *__restrict__ rmap,
                                                       const unsigned short *__restrict__ cb,
                                                       const int *__restrict__ nbase, const int *__restrict__ off,
                                                       const T *__restrict__ vals, const T *__restrict__ xin,
                                                       int nslice, Epi epi, const KStateT<T> *st) {
  if (st && solve_done(st)) return;
  spmv_sellb_body<T, T, BS, U, D>(rows, n, rmap, cb, nbase, off, vals, xin, nslice, epi);
}

template <typename T, int D, class Epi>
static void launch_epi_sellb(ehip_system *s, const T *sv, const T *xin, const Epi &e, const KStateT<T> *st) {
  const int g = sell_grid(s);
  if (s->prof_start)
    hipExtLaunchKernelGGL((k_spmv_epi_sellb<T, 256, kSellBU, D, Epi>), dim3(g), dim3(256), 0, s->stream,
                          s->prof_start, s->prof_stop, 0, s->rows, s->n, s->sell_row, s->sellb_c16, s->sellb_base,
                          s->sell_off, sv, xin, s->nslice, e, st);
  else
    launch_k((k_spmv_epi_sellb<T, 256, kSellBU, D, Epi>), dim3(g), dim3(256), s->stream, s->rows, s->n, s->sell_row,
             s->sellb_c16, s->sellb_base, s->sell_off, sv, xin, s->nslice, e, st);
}

// Workgroups of an epilogue SpMV on the SELL-64 layout: sell_grid, but at
// most 1024 for the FP32 plain-SELL kernels, whose waves then take ~8 slices
// each and spread their per-slice epilogue set-up (and the vector step
// after them reduces 4x fewer partials): the fused FP32 CG step on 128^3
// Hex8 Poisson measured 73.5 against 75.2 us.  The FP64 and node-blocked
// kernels measured slower that way and keep sell_grid.
// On the half storage, whose step takes its second reads from the caches
// and gains from more waves in flight, 2048: whole mixed solves with 1024 /
// 2048 / 3072 / 4096 workgroups take 12.3 / 12.0 / 12.4 / 12.7 ms at 101^3 and
// 25.5 / 24.6 / 24.4 / 24.9 ms at 128^3 (beyond 2048 the vector step, whose
// workgroups each add up all partial sums, loses what the SpMV gains).
template <typename T>
static int epi_sell_grid(const ehip_system *s, bool half = false) {
  if (sizeof(T) != 4 || s->sellb_d) return sell_grid(s);
  return std::min(sell_grid(s), half ? 2048 : 1024);
}

template <int U, class Epi>
static void launch_epi_sell2(ehip_system *s, const double *sv, const double *xin, const Epi &e, const KState *st) {
  const int g = sell_grid(s);
  if (s->prof_start)
    hipExtLaunchKernelGGL((k_spmv_epi_sell2<256, U, Epi>), dim3(g), dim3(256), 0, s->stream, s->prof_start,
                          s->prof_stop, 0, s->rows, s->n, s->sell_row, s->sell2_c16, s->sell_base, s->sell2_off, sv,
                          xin, s->nslice, e, st);
  else
    launch_k((k_spmv_epi_sell2<256, U, Epi>), dim3(g), dim3(256), s->stream, s->rows, s->n, s->sell_row,
             s->sell2_c16, s->sell_base, s->sell2_off, sv, xin, s->nslice, e, st);
}

template <typename T, int U, bool C16, class Epi>
static void launch_epi_sell(ehip_system *s, const T *sv, const T *xin, const Epi &e, const KStateT<T> *st) {
  const int g = epi_sell_grid<T>(s);
  if (s->prof_start)
    hipExtLaunchKernelGGL((k_spmv_epi_sell<T, 256, U, C16, Epi>), dim3(g), dim3(256), 0, s->stream, s->prof_start,
                          s->prof_stop, 0, s->rows, s->n, s->sell_row, s->sell_c32, s->sell_c16, s->sell_base,
                          s->sell_off, sv, xin, s->nslice, e, st);
  else
    launch_k((k_spmv_epi_sell<T, 256, U, C16, Epi>), dim3(g), dim3(256), s->stream, s->rows, s->n, s->sell_row,
             s->sell_c32, s->sell_c16, s->sell_base, s->sell_off, sv, xin, s->nslice, e, st);
}

template <typename T, int U, int D, bool NT, class Epi>
static void launch_epi_sho_as(ehip_system *s, const T *sv, const T *xin, const Epi &e, const KStateT<T> *st) {
  const int g = epi_sell_grid<T>(s);
  const int nt_from = sho_nt_from(s->nslice, (int64_t)sizeof(T) * s->sho_nnz, s->n, (int)sizeof(T));
  if (s->prof_start)
    hipExtLaunchKernelGGL((k_spmv_epi_sho<T, 256, U, D, NT, Epi>), dim3(g), dim3(256), 0, s->stream, s->prof_start,
                          s->prof_stop, 0, s->n, s->sho_off, s->sho_tab, s->sho_mask, sv, xin, s->nslice, nt_from, e,
                          st);
  else
    launch_k((k_spmv_epi_sho<T, 256, U, D, NT, Epi>), dim3(g), dim3(256), s->stream, s->n, s->sho_off, s->sho_tab,
             s->sho_mask, sv, xin, s->nslice, nt_from, e, st);
}

template <typename T, int U, int D, class Epi>
static void launch_epi_sho(ehip_system *s, const T *sv, const T *xin, const Epi &e, const KStateT<T> *st) {
  if (sho_streamed((int64_t)sizeof(T) * s->sho_nnz)) launch_epi_sho_as<T, U, D, true>(s, sv, xin, e, st);
  else launch_epi_sho_as<T, U, D, false>(s, sv, xin, e, st);
}

// Epilogues that run on the half storage too: those of the CG loops
// (ehip_system::sym_on is set for these solves only).
template <class Epi>
struct EpiOnSym : std::false_type {};
template <typename T> struct EpiOnSym<EpiInit<T>> : std::true_type {};
template <typename T> struct EpiOnSym<EpiTrue<T>> : std::true_type {};
template <typename T> struct EpiOnSym<EpiCgQ<T>> : std::true_type {};
template <typename T> struct EpiOnSym<EpiCgResidual<T>> : std::true_type {};
template <typename T> struct EpiOnSym<EpiCgFast1<T>> : std::true_type {};
template <typename T> struct EpiOnSym<EpiCgFold<T>> : std::true_type {};
template <> struct EpiOnSym<EpiRU> : std::true_type {};
template <> struct EpiOnSym<EpiResid> : std::true_type {};

template <typename T, int BS, int U, int D, class Epi>
__global__ __launch_bounds__(BS) void k_spmv_epi_sym(int n, SymTab tab, const unsigned long long *__restrict__ pm,
                                                     const unsigned long long *__restrict__ zero,
                                                     const T *__restrict__ vals, const T *__restrict__ xin, int nslice,
                                                     Epi epi, const KStateT<T> *st) {
  if (st && solve_done(st)) return;
  spmv_sym_body<T, T, BS, U, D>(n, tab, pm, zero, vals, xin, nslice, epi);
}

template <typename T, int D, class Epi>
static void launch_epi_sym(ehip_system *s, const T *sv, const T *xin, const Epi &e, const KStateT<T> *st) {
  const int g = epi_sell_grid<T>(s, true);
  const unsigned long long *zero;
  if constexpr (sizeof(T) == 4) zero = s->sym32.zero; else zero = s->sym64.zero;
  if (s->prof_start)
    hipExtLaunchKernelGGL((k_spmv_epi_sym<T, 256, 9, D, Epi>), dim3(g), dim3(256), 0, s->stream, s->prof_start,
                          s->prof_stop, 0, s->n, s->sym_tab, s->sym_pm, zero, sv, xin, s->nslice, e, st);
  else
    launch_k((k_spmv_epi_sym<T, 256, 9, D, Epi>), dim3(g), dim3(256), s->stream, s->n, s->sym_tab, s->sym_pm, zero, sv,
             xin, s->nslice, e, st);
}

// the active format of one precision: 0 CSR stream, 1 SELL-64, 2 SELL-64
// with slice-shared offsets
template <typename T>
static int active_fmt(const ehip_system *s) {
  const int f = sizeof(T) == 4 ? s->fmt32 : s->fmt64;
  return f == 2 ? (s->sho_ok ? 2 : 0) : (f == 1 && s->sell_ok ? 1 : 0);
}

// Workgroups (and so published partials) of the epilogue SpMV launch last
// enqueued: the half storage's when that copy holds the current values
template <typename T>
static int epi_grid(const ehip_system *s, const SpmvPlan &p) {
  const int fmt = active_fmt<T>(s);
  if (!fmt) return p.grid;
  if constexpr (sizeof(T) == 4)
    return epi_sell_grid<T>(s, fmt == 2 && (s->sym_on & 2) && s->sym32.good && s->sym32.ver == s->vals32_ver);
  return epi_sell_grid<T>(s);
}

// SpMV with epilogue on the system's active format (SELL-64 or CSR stream);
// `vals` names the CSR values (FP64 Values or the FP32 copy) whose SELL
// copy is used in the SELL format.
template <typename T, class Epi>
static void launch_epi(ehip_system *s, const SpmvPlan &p, const T *vals, const T *xin, const Epi &e,
                       const KStateT<T> *st) {
  constexpr bool F32 = sizeof(T) == 4;
  // a values copy that could not be allocated: no launch, the driver's
  // take_launch_error() check ends the solve
  auto missing = [](const void *sv) {
    if (sv) return false;
    if (tl_launch_err == hipSuccess) tl_launch_err = hipErrorOutOfMemory;
    return true;
  };
  if (active_fmt<T>(s) == 2) {
    const T *sv;
    if constexpr (EpiOnSym<Epi>::value) {
      if constexpr (F32) sv = sym_values32(s); else sv = sym_values64(s);
      if (sv) {
        s->route_half |= F32 ? 2 : 1;
        if (s->sho_d == 3) launch_epi_sym<T, 3>(s, sv, xin, e, st);
        else launch_epi_sym<T, 1>(s, sv, xin, e, st);
        return;
      }
    }
    if constexpr (F32) sv = sho_values32(s); else sv = sho_values64(s);
    if (missing(sv)) return;
    if (s->sho_d == 3) launch_epi_sho<T, 9, 3>(s, sv, xin, e, st);
    else if (s->sho_d == 2) launch_epi_sho<T, 9, 2>(s, sv, xin, e, st);
    else if (s->sho_u == 9) launch_epi_sho<T, 9, 1>(s, sv, xin, e, st);
    else launch_epi_sho<T, 8, 1>(s, sv, xin, e, st);
    return;
  }
  if (active_fmt<T>(s) == 1) {
    const T *sv;
    if constexpr (F32) sv = sell_values32(s); else sv = sell_values64(s);
    if (missing(sv)) return;
    if (s->sellb_d) {  // node-blocked layout
      if (s->sellb_d == 3) launch_epi_sellb<T, 3>(s, sv, xin, e, st);
      else launch_epi_sellb<T, 2>(s, sv, xin, e, st);
      return;
    }
    if constexpr (!F32) {
      if (s->sell2_ok) {  // pair-packed FP64 layout
        if (s->sell2_u == 7) launch_epi_sell2<7>(s, sv, xin, e, st);
        else launch_epi_sell2<kSell2U>(s, sv, xin, e, st);
        return;
      }
    }
    // a sampled launch carries its timing events (s->prof_start/stop); other
    // launches -- including those recorded into graphs -- are plain launches
    if (s->sell_u == 9) {
      if (s->sell_c16) launch_epi_sell<T, 9, true>(s, sv, xin, e, st);
      else launch_epi_sell<T, 9, false>(s, sv, xin, e, st);
    } else {
      if (s->sell_c16) launch_epi_sell<T, kSellU, true>(s, sv, xin, e, st);
      else launch_epi_sell<T, kSellU, false>(s, sv, xin, e, st);
    }
    return;
  }
  if (s->c16)
    launch_epi_cs<T, ColsU16>(s, p, vals, xin, e, st);
  else
    launch_epi_cs<T, ColsI32>(s, p, vals, xin, e, st);
}

// SpMV with epilogue, then its one-workgroup finalize
template <typename T, class Epi>
static void launch_epi_fin(ehip_system *s, const SpmvPlan &p, const T *vals, const T *xin, const Epi &e,
                           const KStateT<T> *st) {
  launch_epi<T, Epi>(s, p, vals, xin, e, st);
  if constexpr (Epi::NV > 0) launch_k((k_fin<T, Epi>), dim3(1), dim3(256), s->stream, e, epi_grid<T>(s, p), st);
}

// vector kernel's finalize
template <typename T, class Fin>
static void fin(ehip_system *s, const Fin &f, int g, const KStateT<T> *st) {
  launch_k((k_fin<T, Fin>), dim3(1), dim3(256), s->stream, f, g, st);
}

// *out = sum of (x_i / d_i)^2, or of x_i^2 without d (two launches, no
// in-kernel fence)
static void sumsq(ehip_system *s, int n, const double *x, double *out, const double *d = nullptr) {
  const int g = vec_grid(n);
  hipLaunchKernelGGL(k_sumsq, dim3(g), dim3(kVecBlock), 0, s->stream, n, x, d, s->partials, (unsigned *)nullptr,
                     (double *)nullptr);
  hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(256), 0, s->stream, s->partials, g, out);
}

template <typename T>
static int read_state(ehip_system *s, KStateT<T> *dst, KStateT<T> *hst) {
  EHIP_HIP_TRY(hipMemcpyAsync(hst, dst, sizeof(KStateT<T>), hipMemcpyDeviceToHost, s->stream));
  EHIP_HIP_TRY(hipStreamSynchronize(s->stream));
  return EHIP_OK;
}

struct SolveCtx {
  int method, precond, maxit, check, mode;
  bool check_set;  // check_every given by the caller (else the loops choose)
  double tol, divtol;
  double tol_u;        // unscaled-residual tolerance (0: HUTI's scaled test alone)
  const double *du;    // the scaling's D when tol_u > 0 (FP64 loops only)
  double *hist;  // device, may be null
  int spmv;
  bool prof;     // sample the SpMV launches of this loop
  DeviceUse *use;
};

template <typename T>
static Vecs<T> make_vecs(T *w, int n, int method, T *x, T *b) {
  Vecs<T> v{};
  const size_t N = (size_t)n;
  v.x = x;
  v.b = b;
  if (method == EHIP_CG) {
    v.r = w; v.z = w + N; v.p = w + 2 * N; v.q = w + 3 * N; v.t = w + 4 * N; v.dg = w + 5 * N;
  } else {
    v.r = w; v.rtld = w + N; v.p = w + 2 * N; v.t1v = w + 3 * N; v.v = w + 4 * N;
    v.sv = w + 5 * N; v.t2v = w + 6 * N; v.t = w + 7 * N; v.dg = w + 8 * N; v.z = w + 9 * N;
  }
  return v;
}
static int nvecs(int method) { return method == EHIP_CG ? 6 : 10; }

// A Krylov sequence in one launch (resident.hip), until it stops or the launch
// has run its number of iterations (hst->done tells); its state in hst.
// *resident = false: there was no room for it, or the grid gave up waiting
// (the device is shared with something that kept part of it off the chip),
// and the vectors and the state are as before, for the launched loop to go
// on from.
template <typename T>
static int run_resident(ehip_system *s, SolveCtx &c, const Vecs<T> &v, KStateT<T> *st, KStateT<T> *hst, bool faithful,
                        double *hist, const T *du, int it0, bool *resident) {
  const int g = resident_groups(s->n, c.method == EHIP_CG);
  // no memory for the buffers, which the launched loop does without; or others
  // hold the chip, or use it
  if (!resident_buffers(s) || !resident_admit(s, g)) {
    *resident = false;
    c.use->launch();
    return EHIP_OK;
  }
  int rc = (c.method == EHIP_CG ? resident_cg<T> : resident_bicgstab<T>)(s, v, st, faithful, hist, du);
  if (!rc) rc = read_state(s, st, hst);
  resident_release(s, g, !rc && hst->ticket[3] != 0);
  if (rc) return rc;
  *resident = hst->ticket[3] == 0;
  s->route_loops |= *resident ? EHIP_LOOP_RESIDENT : EHIP_LOOP_GAVE_UP;
  if (!*resident) c.use->launch();
  if (*resident) c.spmv += std::max(0, hst->iter - it0) * ((faithful ? 2 : 1) + (c.method == EHIP_CG ? 0 : 1));
  return EHIP_OK;
}

// Krylov iterations on a scaled system in precision T.  For T = double the
// vectors are s->x / s->rhs; for the FP32 inner solve of the mixed form they
// are the caller's.  Returns with the final state in hst.
template <typename T>
static int krylov(ehip_system *s, SolveCtx &c, const SpmvPlan &plan, const T *vals, Vecs<T> v,
                  KStateT<T> *st, KStateT<T> *hst, T *part, bool init_residual) {
  const int n = s->n;
  const int g = vec_grid(n);
  const int gf = fused_grid(n);
  const int pg = kEpiStride;
  int rc;
  const int iter0 = (c.mode == EHIP_FAITHFUL || c.method == EHIP_BICGSTAB) ? 1 : 0;
  // the unscaled test runs on FP64 residuals only
  const T *du = std::is_same<T, double>::value ? reinterpret_cast<const T *>(c.du) : nullptr;
  const T tol_u = du ? (T)c.tol_u : (T)0;
  if (init_residual) {
    hipLaunchKernelGGL(k_init_state<T>, dim3(1), dim3(1), 0, s->stream, st, (T)c.tol, c.maxit, (T)c.divtol, iter0,
                       tol_u);
    EpiInit<T> e{v, st, part, pg, &st->ticket[0]};
    launch_epi_fin<T>(s, plan, vals, v.x, e, (const KStateT<T> *)nullptr);
    c.spmv++;
  } else {
    // mixed inner solve: k_to32 prepared r, z, rho; x (= d) is zero
    hipLaunchKernelGGL(k_init_state<T>, dim3(1), dim3(1), 0, s->stream, st, (T)c.tol, c.maxit, (T)c.divtol, iter0,
                       tol_u);
  }
  bool resident = s->resident_on && resident_fits<T>(s, c.method == EHIP_CG, c.mode == EHIP_FAITHFUL);
  if (c.method == EHIP_CG) {
    if (c.mode == EHIP_FAITHFUL) {
      EHIP_HIP_TRY(hipMemcpyAsync(v.p, v.z, sizeof(T) * n, hipMemcpyDeviceToDevice, s->stream));
      for (int it_seen = iter0; resident; it_seen = hst->iter) {
        if ((rc = run_resident<T>(s, c, v, st, hst, true, c.hist, du, it_seen, &resident))) return rc;
        if (hst->done) break;
      }
      for (; !resident;) {
        s->route_loops |= EHIP_LOOP_LAUNCHED;
        for (int k = 0; k < c.check; ++k) {
          EpiCgQ<T> e1{v, st, part, pg, &st->ticket[0]};
          if (c.prof) prof_begin(s);
          launch_epi<T>(s, plan, vals, v.p, e1, st);
          if (c.prof) prof_end(s);
          hipLaunchKernelGGL(k_cg_da<T>, dim3(gf), dim3(kVecBlock), 0, s->stream, n, v, st, (const T *)part,
                             epi_grid<T>(s, plan), part + kVecPartOff);
          EpiCgResidual<T> e2{v, st, part, pg, &st->ticket[2], c.hist, part + kVecPartOff, gf, (T)0, du};
          launch_epi_fin<T>(s, plan, vals, v.x, e2, st);
          c.spmv += 2;
        }
        if ((rc = read_state(s, st, hst))) return rc;
        if (hst->done) break;
      }
    } else {
      hipLaunchKernelGGL(k_zero2<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v.p, v.q);
      for (int it_seen = iter0;; it_seen = hst->iter) {
        if (resident && (rc = run_resident<T>(s, c, v, st, hst, false, c.hist, du, it_seen, &resident))) return rc;
        if (!resident) s->route_loops |= EHIP_LOOP_LAUNCHED;
        for (int k = 0; !resident && k < c.check; ++k) {
          EpiCgFast1<T> e1{v, st, part, pg, &st->ticket[0], (T)0};
          if (c.prof) prof_begin(s);
          launch_epi<T>(s, plan, vals, v.z, e1, st);
          if (c.prof) prof_end(s);
          hipLaunchKernelGGL(k_cg_fast2<T>, dim3(gf), dim3(kVecBlock), 0, s->stream, n, v, st, (const T *)part,
                             epi_grid<T>(s, plan), part + kVecPartOff);
          fin<T>(s, FinCgFast2<T>{st, part + kVecPartOff, gf, c.hist}, gf, st);
          c.spmv++;
        }
        if (!resident && (rc = read_state(s, st, hst))) return rc;
        if (!hst->done) continue;
        if (!hst->rec_conv || !init_residual) break;  // inner solves stop on the recurrence
        // recurrence converged: confirm with the true residual, restart from it otherwise
        EpiTrue<T> et{v, st, part, pg, &st->ticket[0], du};
        launch_epi_fin<T>(s, plan, vals, v.x, et, (const KStateT<T> *)nullptr);
        c.spmv++;
        if ((rc = read_state(s, st, hst))) return rc;
        if (hst->done) break;
      }
    }
  } else {
    hipLaunchKernelGGL(k_bi_start<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st, part);
    fin<T>(s, FinBiStart<T>{st, part, g}, g, st);
    for (int it_seen = iter0;; it_seen = hst->iter) {
      if (resident &&
          (rc = run_resident<T>(s, c, v, st, hst, c.mode == EHIP_FAITHFUL, c.hist, du, it_seen, &resident)))
        return rc;
      if (!resident) s->route_loops |= EHIP_LOOP_LAUNCHED;
      for (int k = 0; !resident && k < c.check; ++k) {
        EpiBiV<T> e3{v, st, part, pg, &st->ticket[0]};
        if (c.prof) prof_begin(s);
        launch_epi<T>(s, plan, vals, v.t1v, e3, st);
        if (c.prof) prof_end(s);
        fin<T>(s, e3, epi_grid<T>(s, plan), st);
        hipLaunchKernelGGL(k_bi_s<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st, part);
        fin<T>(s, FinSnorm<T>{st, part, g}, g, st);
        hipLaunchKernelGGL(k_bi_snorm_exit<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st);
        hipLaunchKernelGGL(k_bi_snorm_mark<T>, dim3(1), dim3(1), 0, s->stream, st);
        EpiBiT<T> e6{v, st, part, pg, &st->ticket[0], 1};
        launch_epi_fin<T>(s, plan, vals, v.t2v, e6, st);
        hipLaunchKernelGGL(k_bi_xr<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st, part,
                           c.mode == EHIP_FAST ? 1 : 0, c.hist);
        fin<T>(s, FinBiXr<T>{st, part, g, c.mode == EHIP_FAST ? 1 : 0, c.hist}, g, st);
        c.spmv += 2;
        if (c.mode == EHIP_FAITHFUL) {
          EpiBiResidual<T> e8{v, st, part, pg, &st->ticket[2], c.hist, (T)0, (T)0, du};
          launch_epi_fin<T>(s, plan, vals, v.x, e8, st);
          c.spmv++;
        } else {
          hipLaunchKernelGGL(k_bi_p<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st);
        }
      }
      if (!resident && (rc = read_state(s, st, hst))) return rc;
      if (!hst->done) continue;
      if (c.mode == EHIP_FAITHFUL || !hst->rec_conv || !init_residual) break;
      EpiTrue<T> et{v, st, part, pg, &st->ticket[0], du};
      launch_epi_fin<T>(s, plan, vals, v.x, et, (const KStateT<T> *)nullptr);
      c.spmv++;
      if ((rc = read_state(s, st, hst))) return rc;
      if (hst->done) break;
      hipLaunchKernelGGL(k_bi_start<T>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st, part);
      fin<T>(s, FinBiStart<T>{st, part, g}, g, st);
    }
  }
  EHIP_HIP_TRY(hipGetLastError());
  EHIP_HIP_TRY(take_launch_error());
  return EHIP_OK;
}

// Mixed precision: FP32 values and vectors, FP32-accumulated inner Krylov
// (fast mode) inside an FP64 iterative refinement on the scaled system.
// FP64 stays on the device only for x, the true residual and its norm.
static int mixed_ir(ehip_system *s, SolveCtx &c, double inner_tol, int inner_maxit, int *inner_total) {
  const int n = s->n;
  int rc;
  const int nv = nvecs(c.method);
  if ((rc = ensure_work(s, 1))) return rc;
  if ((rc = ensure_work32(s, nv + 1))) return rc;
  double *t64 = s->work;
  Vecs<float> v = make_vecs<float>(s->work32, n, c.method, s->work32 + (size_t)nv * n, nullptr);
  v.b = v.r;  // the inner right-hand side is the normalised residual held in r
  const int g = vec_grid(n);
  const int pg = kEpiStride;
  hipLaunchKernelGGL(k_make_dg<float>, dim3(g), dim3(kVecBlock), 0, s->stream, n, s->diag, s->vals, v.dg,
                     c.precond);
  KState *st = s->st;
  // ||b|| of the scaled system and the outer state
  hipLaunchKernelGGL(k_init_state<double>, dim3(1), dim3(1), 0, s->stream, st, c.tol, c.maxit, c.divtol, 0,
                     c.du ? c.tol_u : 0.0);
  sumsq(s, n, s->rhs, &st->rr);
  if ((rc = read_state(s, st, s->h_st))) return rc;
  const double bn = sqrt(s->h_st->rr);
  EHIP_HIP_TRY(hipMemcpyAsync(&st->rhsnorm, &bn, sizeof(double), hipMemcpyHostToDevice, s->stream));
  EHIP_HIP_TRY(hipStreamSynchronize(s->stream));
  *inner_total = 0;
  int outer = 0;
  int bad = 0;             // consecutive inner solves that ended on a non-finite residual
  bool diverged = false;
  SolveCtx ci = c;
  ci.mode = EHIP_FAST;
  ci.hist = nullptr;
  ci.tol = inner_tol;
  ci.divtol = 0;
  ci.tol_u = 0;
  ci.du = nullptr;
  ci.prof = c.prof;
  for (;;) {
    EpiOuter eo{s->rhs, t64, st, s->partials, pg, &st->ticket[0], c.hist, c.du};
    launch_epi_fin<double>(s, s->plan64, s->vals, s->x, eo, (const KState *)nullptr);
    c.spmv++;
    if ((rc = read_state(s, st, s->h_st))) return rc;
    if (s->h_st->done) break;
    if (*inner_total >= c.maxit) break;
    const double scale = s->h_st->scale;
    hipLaunchKernelGGL(k_to32, dim3(g), dim3(kVecBlock), 0, s->stream, n, t64, 1.0 / scale, v.r, v.z, v.x, v.dg,
                       s->st32, s->partials32);
    hipLaunchKernelGGL((k_fin<float, FinTo32>), dim3(1), dim3(256), 0, s->stream, FinTo32{s->st32, s->partials32, g},
                       g, (const KState32 *)nullptr);
    ci.maxit = std::min(inner_maxit, c.maxit - *inner_total);
    ci.spmv = 0;
    if ((rc = krylov<float>(s, ci, s->plan32, s->vals32, v, s->st32, s->h_st32, s->partials32, false))) return rc;
    c.spmv += ci.spmv;
    *inner_total += s->h_st32->iter;
    if (s->h_st32->info == 3) {
      // The inner solve ended on a non-finite residual (FP32 overflow on a
      // hard system): its correction is dropped and the next refinement step
      // restarts from the same FP64 residual with the inner cap halved below
      // the breakdown point (the restart is deterministic, so the same cap
      // would break down the same way).  Three in a row, or a breakdown at
      // the first inner step, end the solve as diverged.
      if (s->h_st32->iter <= 1 || ++bad >= 3) {
        diverged = true;
        break;
      }
      inner_maxit = std::max(1, s->h_st32->iter / 2);
      continue;
    }
    if (s->h_st32->iter == 0) break;  // inner breakdown without progress: stop with the outer residual
    bad = 0;
    hipLaunchKernelGGL(k_correct, dim3(g), dim3(kVecBlock), 0, s->stream, n, s->x, v.x, scale);
    ++outer;
  }
  if ((rc = read_state(s, st, s->h_st))) return rc;
  if (diverged && !s->h_st->done) {
    KState h = *s->h_st;
    h.info = 3;
    h.done = 1;
    *s->h_st = h;
  }
  if (!s->h_st->done) {
    // ran out of iterations
    KState h = *s->h_st;
    h.info = 2;
    h.done = 1;
    *s->h_st = h;
  }
  s->h_st->pad1 = outer;
  s->h_st->iter = *inner_total;
  return EHIP_OK;
}

// Default residual drop between two replacements of the reliable-update CG.
constexpr double kRuDelta = 1e-2;
// Longest block of FP32 iterations between two host checks (graph pieces of
// 32 + 16 + ... iterations).
constexpr int kRuMaxBlock = 63;

// Enqueues `count` FP32 fast-CG iterations of the mixed form: the fused SpMV
// step, the vector step, and the one-workgroup finalize that runs the
// stopping tests after every step (the replacement must follow the step
// that crosses its threshold: running on past it lets the FP32 recurrence
// drift from the true residual, and the continued search direction then
// carries a badly scaled beta).
static void cg32_iterations(ehip_system *s, const Vecs<float> &v, int count, bool prof) {
  const int n = s->n, gf = fused_grid(n), pg = kEpiStride;
  if (!tl_graph_rec) s->route_loops |= EHIP_LOOP_LAUNCHED;
  KState32 *st32 = s->st32;
  float *vpart = s->partials32 + kVecPartOff;
  if (cg_fold_enabled()) {
    // two launches per iteration; the block closes with the last step's finalize
    for (int k = 0; k < count; ++k) {
      EpiCgFold<float> e1{v, st32, s->partials32, pg, &st32->ticket[0], vpart, gf, 0.f, false};
      if (prof) prof_begin(s);
      launch_epi<float>(s, s->plan32, s->vals32, v.z, e1, st32);
      if (prof) prof_end(s);
      launch_k((k_cg_fast2<float, true>), dim3(gf), dim3(kVecBlock), s->stream, n, v, st32,
               (const float *)s->partials32, epi_grid<float>(s, s->plan32), vpart);
    }
    fin<float>(s, FinCgFold<float>{st32, vpart, gf}, gf, st32);
    s->route_grid32 = epi_grid<float>(s, s->plan32);
    return;
  }
  for (int k = 0; k < count; ++k) {
    EpiCgFast1<float> e1{v, st32, s->partials32, pg, &st32->ticket[0], 0.f};
    if (prof) prof_begin(s);
    launch_epi<float>(s, s->plan32, s->vals32, v.z, e1, st32);
    if (prof) prof_end(s);
    launch_k((k_cg_fast2<float>), dim3(gf), dim3(kVecBlock), s->stream, n, v, st32, (const float *)s->partials32,
             epi_grid<float>(s, s->plan32), vpart);
    fin<float>(s, FinCgFast2<float>{st32, vpart, gf, nullptr}, gf, st32);
  }
  s->route_grid32 = epi_grid<float>(s, s->plan32);
}

// The FP32 values that the launched steps of the solve in progress read, in
// the layout they read them (launch_epi), brought up to date; null: no memory.
static const float *cg32_values(ehip_system *s) {
  const int fmt = active_fmt<float>(s);
  if (fmt == 1) return sell_values32(s);
  if (fmt != 2) return s->vals32;
  const float *half = sym_values32(s);
  return half ? half : sho_values32(s);
}

// What a recorded block bakes in: buffers, SpMV layout and schedule.  One
// system may be solved on the half storage and, elsewhere, on the full copy,
// and only the copy in use is up to date; a copy may lie where the other was.
static uint64_t cg32_key(const ehip_system *s, const float *values) {
  const uint64_t parts[] = {(uint64_t)(uintptr_t)s->work32, (uint64_t)(uintptr_t)s->vals32,
                            (uint64_t)(uintptr_t)values, (uint64_t)(values == s->sym32.v),
                            (uint64_t)epi_grid<float>(s, s->plan32),
                            (uint64_t)(uintptr_t)s->partials32,
                            (uint64_t)(uintptr_t)s->st32, (uint64_t)(uintptr_t)s->plan32.chunk_row,
                            (uint64_t)s->fmt32, (uint64_t)s->plan32.block, (uint64_t)s->plan32.nb,
                            (uint64_t)s->plan32.grid, (uint64_t)s->n, (uint64_t)cg_fold_enabled()};
  uint64_t h = 1469598103934665603ull;
  for (uint64_t x : parts) {
    h ^= x;
    h *= 1099511628211ull;
  }
  return h;
}

// Enqueues `count` iterations as replays of recorded blocks (one graph launch
// per power-of-two piece instead of three kernel launches per iteration).  The
// values copy is brought up to date first, outside any recording.  The
// blocks are built node by node (launch_k under a recorder), not captured,
// and hold kernels only; every iteration kernel reads its scalars from the
// device state, so a replay is the same work as direct launches.
static int cg32_iterations_graph(ehip_system *s, const Vecs<float> &v, int count) {
  const float *values = cg32_values(s);
  if (!values) return EHIP_ENOMEM;
  s->route_loops |= EHIP_LOOP_RECORDED;
  if (values == s->sym32.v) s->route_half |= 2;
  s->route_grid32 = epi_grid<float>(s, s->plan32);
  const uint64_t key = cg32_key(s, values);
  if (key != s->cg32_key) {
    // nothing recorded earlier may still be queued when its graph goes
    EHIP_HIP_TRY(hipStreamSynchronize(s->stream));
    for (hipGraphExec_t &g : s->cg32_graph)
      if (g) {
        (void)hipGraphExecDestroy(g);
        g = nullptr;
      }
    s->cg32_key = key;
  }
  for (int b = 5; b >= 0; --b) {
    const int piece = 1 << b;
    while (count >= piece) {
      if (!s->cg32_graph[b]) {
        GraphRec rec;
        EHIP_HIP_TRY(hipGraphCreate(&rec.graph, 0));
        tl_graph_rec = &rec;
        cg32_iterations(s, v, piece, false);
        tl_graph_rec = nullptr;
        hipError_t e = rec.err;
        if (e == hipSuccess) e = hipGraphInstantiate(&s->cg32_graph[b], rec.graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(rec.graph);
        EHIP_HIP_TRY(e);
      }
      EHIP_HIP_TRY(hipGraphLaunch(s->cg32_graph[b], s->stream));
      count -= piece;
    }
  }
  return EHIP_OK;
}

// Mixed-precision CG with reliable updates: one FP32 CG sequence (FP32
// values, vectors and accumulation, fused one-SpMV steps) whose residual is
// replaced by the FP64 true residual b - A x64 each time the FP32 recurrence
// residual has dropped by `delta`; the FP32 solution increment is folded
// into x64 at each replacement.  Unlike restarted refinement the search
// direction survives a replacement, so the iteration count stays that of
// FP64 CG.  Convergence is decided only on the FP64 true residual.
static int mixed_cg_ru(ehip_system *s, SolveCtx &c, double delta, int *inner_total, int *updates) {
  const int n = s->n;
  int rc;
  const int nv = nvecs(EHIP_CG);
  if ((rc = ensure_work32(s, nv + 1))) return rc;
  Vecs<float> v = make_vecs<float>(s->work32, n, EHIP_CG, s->work32 + (size_t)nv * n, nullptr);
  const int g = vec_grid(n);
  const int pg = kEpiStride;
  KState *st = s->st;
  KState32 *st32 = s->st32;
  hipLaunchKernelGGL(k_make_dg<float>, dim3(g), dim3(kVecBlock), 0, s->stream, n, s->diag, s->vals, v.dg,
                     c.precond);
  hipLaunchKernelGGL(k_init_state<double>, dim3(1), dim3(1), 0, s->stream, st, c.tol, c.maxit, c.divtol, 0,
                     c.du ? c.tol_u : 0.0);
  hipLaunchKernelGGL(k_init_state<float>, dim3(1), dim3(1), 0, s->stream, st32, (float)c.tol, c.maxit,
                     (float)c.divtol, 0, 0.f);
  sumsq(s, n, s->rhs, &st->rr);
  hipLaunchKernelGGL(k_set_rhsnorm, dim3(1), dim3(1), 0, s->stream, st, st32);
  hipLaunchKernelGGL(k_zero2<float>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v.p, v.q);
  EpiRU eru{s->rhs, v, st, st32, s->partials, pg, &st->ticket[0], c.hist, delta, c.du};
  launch_epi_fin<double>(s, s->plan64, s->vals, s->x, eru, (const KState *)nullptr);
  c.spmv++;
  int nupd = 0;
  if ((rc = read_state(s, st, s->h_st))) return rc;
  // iterations per check: predicted from the observed convergence rate so
  // that few no-op launches follow the step that asks for a replacement.
  // A check costs a host round trip (tens of microseconds with the device
  // idle) and a no-op iteration past the replacement point a few
  // microseconds, so the prediction aims a little long and, unless the caller
  // fixed check_every, blocks run up to kRuMaxBlock iterations.
  const int cap = c.check_set ? c.check : std::max(c.check, kRuMaxBlock);
  auto predict = [](double iters) { return (int)std::ceil(1.1 * iters) + 2; };
  int it_prev = 0;
  double lres_prev = std::log(std::max(s->h_st->res, 1e-300));
  double rate = 0.0;  // log residual change per iteration (< 0)
  int batch = std::min(cap, 8);
  bool resident = s->resident_on && resident_fits<float>(s, true, false);
  while (!s->h_st->done) {
    if (resident && (rc = run_resident<float>(s, c, v, st32, s->h_st32, false, nullptr, nullptr, it_prev, &resident)))
      return rc;
    if (resident) {
    } else if (c.prof || !graphs_enabled()) {
      cg32_iterations(s, v, batch, c.prof);  // sampled launches need their own events
    } else if ((rc = cg32_iterations_graph(s, v, batch))) {
      return rc;
    }
    if (!resident) {
      c.spmv += batch;
      if ((rc = read_state(s, st32, s->h_st32))) return rc;
    }
    const KState32 h = *s->h_st32;
    if (h.iter > it_prev && h.res > 0.f) {
      const double lr = std::log((double)h.res);
      const double rnew = (lr - lres_prev) / (h.iter - it_prev);
      rate = rate < 0.0 ? 0.5 * (rate + rnew) : rnew;
      it_prev = h.iter;
      lres_prev = lr;
    }
    if (!h.done) {
      // predicted iterations until the replacement threshold, never past maxit
      int want = cap;
      if (rate < 0.0 && h.ru > 0.f && h.res > h.ru) want = predict(std::log((double)h.ru / (double)h.res) / rate);
      batch = std::max(1, std::min({std::max(2, std::min(cap, want)), h.maxit - h.iter}));
      continue;
    }
    // FP32 stopped: replacement due, recurrence converged, or failure
    hipLaunchKernelGGL(k_correct, dim3(g), dim3(kVecBlock), 0, s->stream, n, s->x, v.x, 1.0);
    launch_epi_fin<double>(s, s->plan64, s->vals, s->x, eru, (const KState *)nullptr);
    c.spmv++;
    ++nupd;
    if ((rc = read_state(s, st, s->h_st))) return rc;
    if (s->h_st->done) break;
    if (h.info != 0) {
      // max iterations, divergence or rho = 0 in the FP32 sequence
      s->h_st->info = h.info;
      s->h_st->done = 1;
      break;
    }
    it_prev = h.iter;
    lres_prev = std::log(std::max(s->h_st->res, 1e-300));
    batch = std::max(2, std::min(cap, rate < 0.0 ? predict(std::log(delta) / rate) : cap));
    batch = std::max(1, std::min(batch, h.maxit - h.iter));
  }
  if ((rc = read_state(s, st32, s->h_st32))) return rc;
  EHIP_HIP_TRY(take_launch_error());
  *inner_total = s->h_st32->iter;
  *updates = nupd;
  s->h_st->iter = *inner_total;
  s->h_st->pad1 = nupd;
  return EHIP_OK;
}

// ================================================================ ILU(k)-preconditioned HUTI loops
//
// CG and BiCGStab in huti_cg.src / huti_bicgstab.src order with
// pcondl = CRS_LUPrecondition (u = v, then the LU solve of ilu.hip) and
// pcondr the dummy copy.  The preconditioner dominates each iteration (one
// launch per dependency level, replayed from a recorded graph), so the
// vector steps stay plain kernels and the host checks the state after every
// iteration.  State: rho (this iteration), rho_new (BiCGStab's rho of the
// previous iteration), alpha, beta, omega.

// r = b - A x (and rtld = r for BiCGStab) ; partial b.b
struct EpiIluInit {
  static constexpr int NV = 1;
  EHIP_EPI_MEMBERS(double)
  double *rtld;
  __device__ void init() {}
  struct Pre { double b; };
  __device__ Pre load(int i) const { return Pre{v.b[i]}; }
  __device__ void row(int i, double s, const Pre &pr, double (&acc)[1]) {
    const double ri = pr.b - s;
    v.r[i] = ri;
    if (rtld) rtld[i] = ri;
    acc[0] += pr.b * pr.b;
  }
  __device__ void finish(double (&tot)[1]) {
    if (threadIdx.x == 0) st->rhsnorm = sqrt(tot[0]);
  }
};

// partials of a0.b0 (and a1.b1)
template <int NV>
__global__ __launch_bounds__(kVecBlock) void k_ilu_dots(int n, const double *__restrict__ a0,
                                                        const double *__restrict__ b0, const double *__restrict__ a1,
                                                        const double *__restrict__ b1, double *partials,
                                                        const KState *st) {
  if (solve_done(st)) return;
  double acc[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) acc[k] = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    acc[0] += a0[i] * b0[i];
    if constexpr (NV > 1) acc[1] += a1[i] * b1[i];
  }
  block_publish<double, NV>(acc, partials, gridDim.x);
}

// CG: rho = r.z (HUTI_CG_RHO on zero); beta = rho / rho of the last iteration
struct FinIluCgRho {
  static constexpr int NV = 1;
  KState *st;
  double *partials;
  int stride;
  __device__ void finish(double (&tot)[1]) {
    if (threadIdx.x) return;
    if (tot[0] == 0.0) {
      st->info = 20;
      st->done = 1;
      return;
    }
    st->beta = st->iter > 1 ? tot[0] / st->rho : 0.0;
    st->rho = tot[0];
  }
};

// p = z (first iteration) or z + beta p
__global__ void k_ilu_cg_p(int n, Vecs<double> v, const KState *st) {
  if (solve_done(st)) return;
  const bool first = st->iter == 1;
  const double beta = st->beta;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    v.p[i] = first ? v.z[i] : v.z[i] + beta * v.p[i];
}

// x += alpha p ; r -= alpha q
__global__ void k_ilu_cg_xr(int n, Vecs<double> v, const KState *st) {
  if (solve_done(st)) return;
  const double alpha = st->alpha;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    v.x[i] = v.x[i] + alpha * v.p[i];
    v.r[i] = v.r[i] - alpha * v.q[i];
  }
}

// The stop test: ||A x - b|| / ||b|| (TRESID_SCALED_BYB) and, when on, the
// unscaled residual; then BiCGStab's omega = 0 breakdown, the iteration
// count and the iteration limit in HUTI's order.
struct EpiIluRes {
  static constexpr int NV = 2;
  EHIP_EPI_MEMBERS(double)
  double *hist;
  const double *du;
  int bicg;
  __device__ void init() {}
  struct Pre { double b, d; };
  __device__ Pre load(int i) const { return Pre{v.b[i], du ? du[i] : 1.0}; }
  __device__ void row(int, double s, const Pre &pr, double (&acc)[2]) {
    const double ti = s - pr.b;
    acc[0] += ti * ti;
    const double ui = ti / pr.d;
    acc[1] += ui * ui;
  }
  __device__ void finish(double (&tot)[2]) {
    if (threadIdx.x != 0) return;
    const double res = sqrt(tot[0]) / st->rhsnorm;
    st->res = res;
    const int it = st->iter;
    if (hist && it - 1 < st->maxit) hist[it - 1] = res;
    if (res < st->tol && unscaled_ok(st, tot[1])) {
      st->info = 1;
      st->done = 1;
      return;
    }
    if (bicg) {
      if (st->omega == 0.0) {
        st->info = 37;
        st->done = 1;
        return;
      }
      st->rho_new = st->rho;
    }
    st->iter = it + 1;
    if (it + 1 > st->maxit) {
      st->info = 2;
      st->done = 1;
    }
  }
};

// BiCGStab start: rho of the last iteration 1, omega 1, alpha 0; p = v = 0
__global__ void k_ilu_bi_start(int n, Vecs<double> v, KState *st) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->rho_new = 1.0;
    st->omega = 1.0;
    st->alpha = 0.0;
  }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    v.p[i] = 0.0;
    v.v[i] = 0.0;
  }
}

// rho = rtld.r (HUTI_BICGSTAB_RHO on zero) ; beta = (rho alpha) / (rho_old omega)
struct FinIluBiRho {
  static constexpr int NV = 1;
  KState *st;
  double *partials;
  int stride;
  __device__ void finish(double (&tot)[1]) {
    if (threadIdx.x) return;
    if (tot[0] == 0.0) {
      st->info = 35;
      st->done = 1;
      return;
    }
    st->beta = (tot[0] * st->alpha) / (st->rho_new * st->omega);
    st->rho = tot[0];
  }
};

// p = r + beta (p - omega v)
__global__ void k_ilu_bi_p(int n, Vecs<double> v, const KState *st) {
  if (solve_done(st)) return;
  const double beta = st->beta, omega = st->omega;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    v.p[i] = v.r[i] + beta * (v.p[i] - omega * v.v[i]);
}

// v = A t1v ; alpha = rho / (rtld.v)
struct EpiIluBiV {
  static constexpr int NV = 1;
  EHIP_EPI_MEMBERS(double)
  __device__ void init() {}
  struct Pre { double rt; };
  __device__ Pre load(int i) const { return Pre{v.rtld[i]}; }
  __device__ void row(int i, double s, const Pre &pr, double (&acc)[1]) {
    v.v[i] = s;
    acc[0] += pr.rt * s;
  }
  __device__ void finish(double (&tot)[1]) {
    if (threadIdx.x == 0) st->alpha = st->rho / tot[0];
  }
};

// s = r - alpha v ; partial s.s
__global__ __launch_bounds__(kVecBlock) void k_ilu_bi_s(int n, Vecs<double> v, const KState *st, double *partials) {
  if (solve_done(st)) return;
  const double alpha = st->alpha;
  double acc[1] = {0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double si = v.r[i] - alpha * v.v[i];
    v.sv[i] = si;
    acc[0] += si * si;
  }
  block_publish<double, 1>(acc, partials, gridDim.x);
}

// ||s|| below HUTI_EPSILON: HUTI_BICGSTAB_SNORM after x += alpha t1v
struct FinIluSnorm {
  static constexpr int NV = 1;
  KState *st;
  double *partials;
  int stride;
  __device__ void finish(double (&tot)[1]) {
    if (threadIdx.x) return;
    if (sqrt(tot[0]) < (double)1.17549435E-38f) {  // HUTI_EPSILON (huti_fdefs.h)
      st->snorm_exit = 1;
      st->info = 36;
    }
  }
};

__global__ void k_ilu_bi_snorm_x(int n, Vecs<double> v, const KState *st) {
  if (solve_done(st) || !st->snorm_exit) return;
  const double alpha = st->alpha;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    v.x[i] = v.x[i] + alpha * v.t1v[i];
}

__global__ void k_ilu_bi_snorm_mark(KState *st) {
  if (st->snorm_exit) st->done = 1;
}

// t = A t2v ; omega = (t.s) / (t.t)
struct EpiIluBiT {
  static constexpr int NV = 2;
  EHIP_EPI_MEMBERS(double)
  __device__ void init() {}
  struct Pre { double sv; };
  __device__ Pre load(int i) const { return Pre{v.sv[i]}; }
  __device__ void row(int i, double s, const Pre &pr, double (&acc)[2]) {
    v.t[i] = s;
    acc[0] += s * pr.sv;
    acc[1] += s * s;
  }
  __device__ void finish(double (&tot)[2]) {
    if (threadIdx.x == 0) st->omega = tot[0] / tot[1];
  }
};

// x += alpha t1v + omega t2v ; r = s - omega t
__global__ void k_ilu_bi_xr(int n, Vecs<double> v, const KState *st) {
  if (solve_done(st)) return;
  const double alpha = st->alpha, omega = st->omega;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    v.x[i] = v.x[i] + alpha * v.t1v[i] + omega * v.t2v[i];
    v.r[i] = v.sv[i] - omega * v.t[i];
  }
}

// HUTI CG / BiCGStab preconditioned with ILU(order) of the system's (scaled)
// values, factorized first as IterSolver does (IterSolve.src:418-520).
static int ilu_krylov(ehip_system *s, SolveCtx &c, int order) {
  const int n = s->n;
  int rc;
  if ((rc = ilu_setup(s, order))) return rc;
  if ((rc = ilu_factor(s))) return rc;
  const bool bicg = c.method == EHIP_BICGSTAB;
  Vecs<double> v = make_vecs<double>(s->work, n, c.method, s->x, s->rhs);
  KState *st = s->st;
  const int g = vec_grid(n), pg = kEpiStride;
  double *part = s->partials;
  hipLaunchKernelGGL(k_init_state<double>, dim3(1), dim3(1), 0, s->stream, st, c.tol, c.maxit, c.divtol, 1,
                     c.du ? c.tol_u : 0.0);
  if (bicg) hipLaunchKernelGGL(k_ilu_bi_start, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, st);
  EpiIluInit ei{v, st, part, pg, &st->ticket[0], bicg ? v.rtld : nullptr};
  launch_epi_fin<double>(s, s->plan64, s->vals, v.x, ei, (const KState *)nullptr);
  c.spmv++;
  const KState *chk = st;
  for (;;) {
    if (!bicg) {
      if ((rc = ilu_apply(s, v.r, v.z))) return rc;
      hipLaunchKernelGGL(k_ilu_dots<1>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v.r, v.z, (const double *)nullptr,
                         (const double *)nullptr, part, chk);
      fin<double>(s, FinIluCgRho{st, part, g}, g, chk);
      hipLaunchKernelGGL(k_ilu_cg_p, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, chk);
      EpiCgQ<double> eq{v, st, part, pg, &st->ticket[0]};
      launch_epi_fin<double>(s, s->plan64, s->vals, v.p, eq, chk);
      hipLaunchKernelGGL(k_ilu_cg_xr, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, chk);
      c.spmv++;
    } else {
      hipLaunchKernelGGL(k_ilu_dots<1>, dim3(g), dim3(kVecBlock), 0, s->stream, n, v.rtld, v.r,
                         (const double *)nullptr, (const double *)nullptr, part, chk);
      fin<double>(s, FinIluBiRho{st, part, g}, g, chk);
      hipLaunchKernelGGL(k_ilu_bi_p, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, chk);
      if ((rc = ilu_apply(s, v.p, v.t1v))) return rc;
      EpiIluBiV ev{v, st, part, pg, &st->ticket[0]};
      launch_epi_fin<double>(s, s->plan64, s->vals, v.t1v, ev, chk);
      hipLaunchKernelGGL(k_ilu_bi_s, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, chk, part);
      fin<double>(s, FinIluSnorm{st, part, g}, g, chk);
      hipLaunchKernelGGL(k_ilu_bi_snorm_x, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, chk);
      hipLaunchKernelGGL(k_ilu_bi_snorm_mark, dim3(1), dim3(1), 0, s->stream, st);
      if ((rc = ilu_apply(s, v.sv, v.t2v))) return rc;
      EpiIluBiT et{v, st, part, pg, &st->ticket[0]};
      launch_epi_fin<double>(s, s->plan64, s->vals, v.t2v, et, chk);
      hipLaunchKernelGGL(k_ilu_bi_xr, dim3(g), dim3(kVecBlock), 0, s->stream, n, v, chk);
      c.spmv += 2;
    }
    EpiIluRes er{v, st, part, pg, &st->ticket[0], c.hist, c.du, bicg ? 1 : 0};
    launch_epi_fin<double>(s, s->plan64, s->vals, v.x, er, chk);
    c.spmv++;
    if ((rc = read_state(s, st, s->h_st))) return rc;
    if (s->h_st->done) break;
  }
  EHIP_HIP_TRY(hipGetLastError());
  EHIP_HIP_TRY(take_launch_error());
  return ilu_check(s);
}

// Time marks of a solve: HIP events on the system's stream, or, for callers
// that create no runtime objects, host clock readings taken after the
// stream has drained.
struct SolveClock {
  bool ev = true;
  hipStream_t stream = nullptr;
  hipEvent_t e[4] = {};
  std::chrono::steady_clock::time_point h[4];
  SolveClock(bool use_events, hipStream_t st) : ev(use_events), stream(st) {}
  ~SolveClock() {
    for (hipEvent_t x : e)
      if (x) (void)hipEventDestroy(x);
  }
  hipError_t create() {
    if (!ev) return hipSuccess;
    for (hipEvent_t &x : e) {
      const hipError_t err = hipEventCreate(&x);
      if (err != hipSuccess) return err;
    }
    return hipSuccess;
  }
  hipError_t mark(int i) {
    if (ev) return hipEventRecord(e[i], stream);
    const hipError_t err = hipStreamSynchronize(stream);
    h[i] = std::chrono::steady_clock::now();
    return err;
  }
  // after the last mark has completed
  float ms(int a, int b) const {
    if (!ev) return (float)std::chrono::duration<double, std::milli>(h[b] - h[a]).count();
    float t = 0.f;
    (void)hipEventElapsedTime(&t, e[a], e[b]);
    return t;
  }
};

int solve_impl(ehip_system *s, const ehip_params *p, double *x, ehip_report *r, double *hist, bool events) {
  if (!s || !p) return EHIP_EARG;
  if (int rc0 = assembly_check(s)) return rc0;
  if (!s->has_values) {
    set_error("ehip_solve: the system has no values (assemble or set them first)");
    return EHIP_ESTATE;
  }
  if (p->method != EHIP_CG && p->method != EHIP_BICGSTAB) return EHIP_EARG;
  if (p->maxit < 1 || !(p->tol > 0)) {
    set_error("ehip_solve: maxit must be >= 1 and tol > 0");
    return EHIP_EARG;
  }
  if (p->precond < EHIP_PRECOND_NONE || p->precond > EHIP_PRECOND_ILU0 + 9) {
    set_error("ehip_solve: unknown preconditioner %d", p->precond);
    return EHIP_EARG;
  }
  if (p->precond >= EHIP_PRECOND_ILU0 && p->precision != EHIP_FP64) {
    set_error("ehip_solve: ILU preconditioning runs in FP64 only");
    return EHIP_EUNSUP;
  }
  const int n = s->n;
  int rc;
  if ((rc = ensure_state(s))) return rc;
  s->route_loops = s->route_half = s->route_grid32 = 0;
  struct Leave {  // other callers of the SpMVs here (the engine's reports) have full copies
    ehip_system *s;
    ~Leave() {
      s->sym_on = 0;
      s->resident_on = false;
    }
  } leave{s};
  // half storage only where the method needs a symmetric matrix anyway; the
  // mixed form of 3-DOF node blocks reads no halved FP32 copy, and its FP64
  // products are too few for the check
  s->sym_on = 0;
  if (p->method == EHIP_CG && p->precond < EHIP_PRECOND_ILU0)
    s->sym_on = p->precision == EHIP_FP64 ? sym_pays(s) & 1 : (s->sho_d == 1 ? sym_pays(s) : 0);
  // on a lane, of systems the resident loops would take elsewhere: their
  // copies fit the caches, and the check's wait costs more than it gives
  if (tl_shared_device && s->n <= 262144) s->sym_on = 0;
  // one launch per sequence where the rows fit the chip (not for callers
  // without runtime objects of their own, nor when launches are sampled)
  s->resident_on = events && !tl_shared_device && p->profile_every <= 0 && p->precond < EHIP_PRECOND_ILU0 &&
                   s->resident_test != 1;
  if (s->sym_on && s->resident_on &&
      resident_fits<double>(s, true, p->mode == EHIP_FAITHFUL && p->precision == EHIP_FP64))
    s->sym_on = 0;  // that loop reads the full copy
  const bool cg = p->method == EHIP_CG, fp64 = p->precision == EHIP_FP64;
  DeviceUse use(s->dev, !(s->resident_on && (fp64 ? resident_fits<double>(s, cg, p->mode == EHIP_FAITHFUL)
                                                  : resident_fits<float>(s, cg, false))));
  SolveClock clk(events, s->stream);
  EHIP_HIP_TRY(clk.create());
  ehip_report rep{};
  EHIP_HIP_TRY(clk.mark(0));
  // initial guess
  bool xzero = true;
  if (x) {
    for (int i = 0; i < n && xzero; ++i) xzero = (x[i] == 0.0);
    EHIP_HIP_TRY(hipMemcpyAsync(s->x, x, sizeof(double) * n, hipMemcpyHostToDevice, s->stream));
  } else {
    EHIP_HIP_TRY(hipMemsetAsync(s->x, 0, sizeof(double) * n, s->stream));
  }
  // bnorm and the zero right-hand side exit (SolverUtils.src:7324-7341)
  sumsq(s, n, s->rhs, &s->st->rr);
  if ((rc = read_state(s, s->st, s->h_st))) return rc;
  const double b2 = s->h_st->rr;
  if (!(sqrt(b2) > DBL_MIN)) {
    EHIP_HIP_TRY(hipMemsetAsync(s->x, 0, sizeof(double) * n, s->stream));
    if (x) std::memset(x, 0, sizeof(double) * n);
    rep.info = 1;
    rep.iters = 0;
    rep.norm = 0.0;
    if (r) *r = rep;
    s->has_x = true;
    return EHIP_OK;
  }
  const bool scaling = p->scaling != 0;
  const bool mixed = p->precision == EHIP_MIXED_IR;
  double bscale = 1.0;
  // keep the unscaled b for the report residual
  if ((rc = ensure_work(s, mixed ? 2 : nvecs(p->method) + 1))) return rc;
  double *b0 = s->work + (size_t)(s->nwork - 1) * n;
  EHIP_HIP_TRY(hipMemcpyAsync(b0, s->rhs, sizeof(double) * n, hipMemcpyDeviceToDevice, s->stream));
  if (scaling) {
    if ((rc = scale_system(s, s->rhs, true, s->x, &bscale, mixed))) return rc;
  } else if (mixed) {
    if (!s->vals32)
      if ((rc = dmalloc(s, (void **)&s->vals32, sizeof(float) * s->nnz))) return rc;
    std::vector<double> one(n, 1.0);
    EHIP_HIP_TRY(hipMemcpy(s->dscale, one.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    ScaleValues f{s->vals, s->cols, s->dscale, s->vals32};
    hipLaunchKernelGGL(k_nonzeros<ScaleValues>, dim3(s->plan64.grid), dim3(256), 0, s->stream, s->rows,
                       s->plan64.chunk_row, s->plan64.nchunks, f);
    touch_vals(s, true, true);
  }
  if (xzero)
    hipLaunchKernelGGL(k_fill<double>, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, s->x, 1.0e-8);
  // history buffer
  double *dhist = nullptr;
  if (p->record_history) {
    if (s->hist_cap < p->maxit + 2) {
      if (s->hist) dfree(s, s->hist, sizeof(double) * s->hist_cap);
      s->hist = nullptr;
      s->hist_cap = 0;
      if ((rc = dmalloc(s, (void **)&s->hist, sizeof(double) * (p->maxit + 2)))) return rc;
      s->hist_cap = p->maxit + 2;
    }
    dhist = s->hist;
  }
  SolveCtx c{};
  c.use = &use;
  c.method = p->method;
  c.precond = p->precond;
  c.maxit = p->maxit;
  c.mode = p->mode;
  c.tol = p->tol;
  c.divtol = p->divtol;
  c.check = p->check_every > 0 ? p->check_every : (n > 200000 ? 25 : 10);
  c.check_set = p->check_every > 0;
  c.hist = dhist;
  // the unscaled test: without scaling the scaled residual is the unscaled one
  c.tol_u = (p->true_residual_stop && scaling) ? p->tol : 0.0;
  c.du = c.tol_u > 0 ? s->dscale : nullptr;
  if (c.du) sumsq(s, n, s->rhs, &s->st->bb_u, s->dscale);  // ||b_s / D||^2
  c.prof = p->profile_every > 0;
  s->prof_every = p->profile_every;
  s->prof_n = 0;
  s->prof_count = 0;
  EHIP_HIP_TRY(clk.mark(1));
  int inner_total = 0;
  if (mixed && p->method == EHIP_CG) {
    // reliable-update CG: inner_tol is the residual drop between replacements
    const double delta = p->inner_tol > 0 ? p->inner_tol : kRuDelta;
    int nupd = 0;
    if ((rc = mixed_cg_ru(s, c, delta, &inner_total, &nupd))) return rc;
    rep.outer_iters = nupd;
  } else if (mixed) {
    // restarted refinement: each inner solve reduces the residual by itol.
    // 1e-2 beat 1e-3, 1e-4, 1e-5 and 1e-6 on the convection-diffusion
    // batch (fewer iterations in all: deep FP32 inner solves stagnate)
    const double itol = p->inner_tol > 0 ? p->inner_tol : 1e-2;
    const int imax = p->inner_maxit > 0 ? p->inner_maxit : 1000;
    // FP32 vectors are the workspace; the FP64 workspace holds the residual
    if ((rc = mixed_ir(s, c, itol, imax, &inner_total))) return rc;
    rep.outer_iters = s->h_st->pad1;
  } else if (p->precond >= EHIP_PRECOND_ILU0) {
    s->route_loops = EHIP_LOOP_LAUNCHED;
    if ((rc = ilu_krylov(s, c, p->precond - EHIP_PRECOND_ILU0))) return rc;
  } else {
    Vecs<double> v = make_vecs<double>(s->work, n, p->method, s->x, s->rhs);
    hipLaunchKernelGGL(k_make_dg<double>, dim3(vec_grid(n)), dim3(kVecBlock), 0, s->stream, n, s->diag, s->vals,
                       v.dg, p->precond);
    if ((rc = krylov<double>(s, c, s->plan64, s->vals, v, s->st, s->h_st, s->partials, true))) return rc;
  }
  EHIP_HIP_TRY(clk.mark(2));
  const KState hs = *s->h_st;
  rep.info = hs.info;
  rep.iters = hs.iter;
  rep.res_scaled = hs.res_true >= 0 ? hs.res_true : hs.res;
  if (p->record_history && hist) {
    int k = mixed ? rep.outer_iters + 1 : std::min(hs.iter, p->maxit);
    if (k > 0) EHIP_HIP_TRY(hipMemcpy(hist, dhist, sizeof(double) * k, hipMemcpyDeviceToHost));
  }
  if (scaling)
    if ((rc = backscale_system(s, s->rhs, s->x, bscale))) return rc;
  // unscaled FP64 true residual ||b - A x|| / ||b|| and ComputeNorm
  {
    if (!(s->route_half & 1)) s->sym_on = 0;  // not symmetric when scaled: not asked again
    double *out = reinterpret_cast<double *>(&s->st->ts);
    EpiResid er{b0, s->partials, kEpiStride, &s->st->ticket[0], out};
    launch_epi_fin<double>(s, s->plan64, s->vals, s->x, er, (const KState *)nullptr);
    sumsq(s, n, s->x, &s->st->rr);
    if ((rc = read_state(s, s->st, s->h_st))) return rc;
    rep.res_true = sqrt(s->h_st->ts) / sqrt(s->h_st->tt);
    rep.norm = sqrt(s->h_st->rr / (double)n);
  }
  EHIP_HIP_TRY(clk.mark(3));
  if (x) EHIP_HIP_TRY(hipMemcpyAsync(x, s->x, sizeof(double) * n, hipMemcpyDeviceToHost, s->stream));
  EHIP_HIP_TRY(hipStreamSynchronize(s->stream));
  rep.t_krylov_ms = clk.ms(1, 2);
  rep.t_total_ms = clk.ms(0, 3);
  rep.spmv_count = c.spmv + 1;
  prof_collect(s, &rep.spmv_us, &rep.spmv_samples);
  rep.spmv_precision = mixed ? 1 : 0;
  s->prof_every = 0;
  s->has_x = true;
  if (r) *r = rep;
  return EHIP_OK;
}

}  // namespace ehip

// ================================================================ C ABI

extern "C" int ehip_solve(ehip_system *s, const ehip_params *p, double *x, ehip_report *r, double *hist) {
  return ehip::solve_impl(s, p, x, r, hist, true);
}

extern "C" int ehip_solve_route(const ehip_system *s, int *loops, int *half_storage, int *spmv_grid32) {
  if (!s) return EHIP_EARG;
  if (loops) *loops = s->route_loops;
  if (half_storage) *half_storage = s->route_half;
  if (spmv_grid32) *spmv_grid32 = s->route_grid32;
  return EHIP_OK;
}

extern "C" int ehip_get_solution(ehip_system *s, double *x) {
  if (!s || !x) return EHIP_EARG;
  EHIP_HIP_TRY(hipStreamSynchronize(s->stream));
  EHIP_HIP_TRY(hipMemcpy(x, s->x, sizeof(double) * s->n, hipMemcpyDeviceToHost));
  return EHIP_OK;
}

extern "C" int ehip_solve_csr(int n, const int *rows, const int *cols, const int *diag, const double *values,
                              const double *b, double *x, const ehip_params *p, ehip_report *r) {
  ehip_system *s = nullptr;
  int rc = ehip_system_create(n, (int64_t)rows[n] - 1, rows, cols, diag, &s);
  if (rc) return rc;
  rc = ehip_system_set_values(s, values, b);
  if (!rc) rc = ehip_solve(s, p, x, r, nullptr);
  ehip_system_free(s);
  return rc;
}

// Unscaled FP64 residual ||b0 - A x|| / ||b0|| and ComputeNorm of the
// system's current (back-scaled) solution.
extern "C" int ehip_internal_report(ehip_system *s, const double *b0, double *res_true, double *norm) {
  int rc;
  if ((rc = ensure_state(s))) return rc;
  const int n = s->n;
  double *out = reinterpret_cast<double *>(&s->st->ts);
  EpiResid er{b0, s->partials, kEpiStride, &s->st->ticket[0], out};
  launch_epi_fin<double>(s, s->plan64, s->vals, s->x, er, (const KState *)nullptr);
  sumsq(s, n, s->x, &s->st->rr);
  if ((rc = read_state(s, s->st, s->h_st))) return rc;
  *res_true = sqrt(s->h_st->ts) / sqrt(s->h_st->tt);
  *norm = sqrt(s->h_st->rr / (double)n);
  return EHIP_OK;
}
