// Resident Krylov loops: a whole CG sequence of a system of moderate size in
// one launch.
//
// Below a quarter of a million rows an iteration of the launched loops
// (krylov.hip) is bound by its two to four dependent launches of 4 to 8 us
// each, not by the matrix: 27 us an iteration in HUTI's order on 17^3 Hex8
// (5 832 rows), 21 us for the one-SpMV order on 47^3.  Here every row belongs
// to one thread of a grid that stays on the chip until the sequence stops:
// the thread's entries of x, r, z, p, q and the Jacobi diagonal stay in its
// registers, the matrix in the L2 of its XCD, and the vector that the SpMV
// gathers in the workgroup's LDS (its 1024 rows and a halo of the
// bandwidth).  What is left of an iteration are its two exchanges between
// workgroups (four in BiCGStab): partial sums, and the halo's new entries with
// the second one.  Per iteration, launched and resident: 17^3 Hex8 in HUTI's
// order 27 and 10 us, 55^3 Tet4 (SELL-64) one-SpMV order 20 and 17 us, 301^2
// Quad4 BiCGStab in HUTI's order 52 and 25 us.  Of the 10 us, measured by the
// kernel's own clock, some 5 are the exchanges' trips to the memory the XCDs
// share, the rest the row sums and the reductions inside the workgroup.
//
// Exchanges.  A workgroup publishes its partial sums as 64-bit words that
// carry the exchange's number beside 32 bits of the value, with agent-scope
// stores; everyone polls the words of all workgroups and adds them up in the
// launched loops' order.  Vector entries go out before that with
// agent-scope stores, acknowledged before the partial sums are published,
// and are read with agent-scope loads after everyone's have been seen: no
// cache is written back or invalidated.  The words of one exchange are
// written again two exchanges later, when every workgroup has published the
// one between and so has read them.
//
// Bits.  Sums are grouped as the launched kernels group them -- the SpMV's
// partials per 256 rows, CG's vector step's per 1024 rows with four rows to
// a thread, the totals over 256 threads -- and the scalar updates and
// stopping tests are the same functors (cg_steps.h), so a solve gives the
// same bits either way.  BiCGStab's launched vector steps walk the rows by
// a grid of G = vec_grid workgroups, so a partial sum there takes the tiles
// of 256 rows b, b + G, b + 2 G and b + 3 G, a thread one row of each: a
// resident workgroup owns those four tiles, each with its window, instead
// of 1024 rows in a row.  (Its solutions near the s-norm exit follow the
// order of the sums by far more than rounding, so another grouping would be
// another answer.)  That takes three more halos: of FP64 systems, a bandwidth
// up to 920 fits the LDS (1 970 with one window) where CG's 1024 rows in a
// row take 3 680 (7 880).
//
// Waiting.  All workgroups of the grid must be on the chip at once.  A
// workgroup (1024 threads of at most 128 registers, at most 156 of 160 KB of
// LDS) fits any CU that no other one holds, so the process counts CUs: loops
// run side by side while every XCD has a CU for each workgroup of theirs that
// it can be given (resident_admit); one that finds no room runs launched.
// Beside launched kernels none is started: a loop keeps the CUs, and a
// hardware queue that streams may share, from them until it stops, where
// launched loops take turns kernel by kernel.  For the same reason a launch
// stops after kSlice iterations (kSliceShared when other solves are in
// progress), so whoever comes then waits for no more than those.
// Other kernels end by themselves, and every wait is bounded: a thread that
// polls past kSpins (a quarter of a second or so) gives up for the whole
// grid.  That is for what the count does not see, other processes and CU
// masks; it does not happen again for kRest.  Results go to separate
// buffers, which a commit launch copies only if nobody gave up, so the
// launched loop then takes over from the unchanged vectors.
#include <hip/hip_runtime.h>

#include <chrono>
#include <mutex>

#include "cg_steps.h"
#include "ehip_internal.h"
#include "launch.h"

namespace ehip {

namespace {

constexpr int kResRows = 1024;    // rows (and threads) of a workgroup
constexpr int kResGroups = 256;   // at most, one per CU
constexpr int kResLds = 156 * 1024;
constexpr int kSpins = 1 << 18;
constexpr int kCusPerXcd = 32;
// Iterations of a launch: 2 to 12 ms, against some 40 us to go on with the
// next, and 0.3 to 1.5 ms.
constexpr int kSlice = 256, kSliceShared = 32;
typedef unsigned long long Word;

__device__ __forceinline__ Word ld_word(const Word *p) {
  return __hip_atomic_load(const_cast<Word *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_word(Word *p, Word v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_agent(const double *p) {
  return __hip_atomic_load(const_cast<double *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_agent(const float *p) {
  return __hip_atomic_load(const_cast<float *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// this wave's stores have reached the coherence point
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A value as words: FP32 one, FP64 two.
template <typename T>
constexpr int kWords = sizeof(T) / 4;
__device__ __forceinline__ void publish(Word *p, unsigned e, double v) {
  const Word b = (Word)__double_as_longlong(v), hi = (Word)e << 32;
  st_word(p, hi | (b & 0xffffffffull));
  st_word(p + 1, hi | (b >> 32));
}
__device__ __forceinline__ void publish(Word *p, unsigned e, float v) {
  st_word(p, ((Word)e << 32) | __float_as_uint(v));
}
__device__ __forceinline__ bool seen(const Word *p, unsigned e, double &v) {
  const Word a = ld_word(p), b = ld_word(p + 1);
  v = __longlong_as_double((long long)((a & 0xffffffffull) | (b << 32)));
  return (unsigned)(a >> 32) == e && (unsigned)(b >> 32) == e;
}
__device__ __forceinline__ bool seen(const Word *p, unsigned e, float &v) {
  const Word a = ld_word(p);
  v = __uint_as_float((unsigned)a);
  return (unsigned)(a >> 32) == e;
}

}  // namespace

namespace {

// wave_sum (reduce.h) with the last four steps as rotations inside rows of
// 16 lanes instead of cross-lane LDS operations: after the steps of 32 and
// 16 lanes the sums repeat every 16, 8, ... lanes, so adding the lane 8, 4,
// 2, 1 further on adds the same two numbers (the same bits).
template <int CTRL>
__device__ __forceinline__ float rotated(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double rotated(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((Word)hi << 32) | lo));
}
template <typename T>
__device__ __forceinline__ T row_wave_sum(T v) {
  v += __shfl_xor(v, 32, kWave);
  v += __shfl_xor(v, 16, kWave);
  v += rotated<0x128>(v);  // row_ror:8
  v += rotated<0x124>(v);
  v += rotated<0x122>(v);
  v += rotated<0x121>(v);
  return v;
}

}  // namespace

// The matrix in the layout the launched SpMV reads: slice-shared offsets
// (SHO), or SELL-64 with 16-bit columns, FP64 values pair-packed.
enum ResFmt { RES_SHO, RES_SELL };

template <typename T>
struct ResArgs {
  int n, nslice, halo;
  int ngroups;                  // 256-row groups with rows
  int spmv_grid, vec_grid;      // workgroups of the launched kernels
  int cap;                      // iterations after which the launch stops
  const int *off, *tab;         // SHO: slice offsets and offset lists; SELL: slice offsets, slice bases
  const unsigned *mask;         // SHO
  const unsigned short *c16;    // SELL
  const int *rows;              // SELL
  const T *vals;
  Vecs<T> v, out;               // the vectors, and where the results go
  const KStateT<T> *st;
  KStateT<T> *st_out;
  Word *w1, *w2;                // words of the two exchanges
  T *ex, *ez, *er, *ew;         // vector entries on their way to other workgroups
  int *gave_up;
  double *hist;
  const T *du;
};

namespace {

// launched workgroup of the SpMV that has 256-row group g (XcdWalk: at most
// one group each, the grid being at least as large as their number)
__device__ __forceinline__ int spmv_slot(int g, int ngroups) {
  int xcd = (int)((long long)g * 8 / ngroups);
  while ((long long)ngroups * (xcd + 1) / 8 <= g) ++xcd;
  while ((long long)ngroups * xcd / 8 > g) --xcd;
  return (g - (int)((long long)ngroups * xcd / 8)) * 8 + xcd;
}
// The slot of the group that this thread publishes, -1 where it has no rows;
// found once, as it takes a division.
__device__ __forceinline__ int group_slot(int g, int ngroups) { return g < ngroups ? spmv_slot(g, ngroups) : -1; }
__device__ __forceinline__ bool slot_used(int b, int ngroups) {
  const int xcd = b & 7, lb = b >> 3;
  return (int)((long long)ngroups * xcd / 8) + lb < (int)((long long)ngroups * (xcd + 1) / 8);
}

// A row's matrix entries.  SHO: the values in registers (at most KW of
// them), the slice's offset list in scalar loads of many offsets each (one
// by one, each cost its latency: 5.7 us of a 15 us iteration at 17^3 Hex8).
// SELL: read from the L2 in every product.
template <typename T, ResFmt F, int KW>
struct ResRow {
  T v[F == RES_SHO ? KW : 1];
  unsigned m;  // SHO: the row's own entries (FP32: all of the list's)
  int wd, p0, len;
  __device__ __forceinline__ void load(const ResArgs<T> &a, int sl, int lane) {
    constexpr bool kF32 = sizeof(T) == 4;
    const int r = sl * 64 + lane;
    const int rl = min(r, a.n - 1);
    const bool live = sl < a.nslice;
    p0 = live ? a.off[sl] : 0;
    const int width = live ? a.off[sl + 1] - p0 : 0;
    if constexpr (F == RES_SHO) {
      wd = width >> 6;
      m = kF32 ? (wd >= 32 ? ~0u : (1u << wd) - 1u) : (r < a.n ? a.mask[rl] : 0u);
#pragma unroll
      for (int k = 0; k < KW; ++k) v[k] = k < wd ? a.vals[p0 + 64 * k + lane] : (T)0;
    } else {
      wd = kF32 ? width >> 6 : width >> 7;
      len = r < a.n ? a.rows[rl + 1] - a.rows[rl] : 0;
    }
  }
  // Sums of one or two vectors held in LDS windows starting at column wb, in
  // the launched kernels' order (spmv_sho_body, spmv_sell2_body,
  // spmv_sell_body).
  // `own` is the row's own place there.
  template <int NX>
  __device__ __forceinline__ void sums(const ResArgs<T> &a, int sl, int lane, int wb, int own, const T *w0,
                                       const T *w1, T (&s)[NX]) const {
    constexpr bool kF32 = sizeof(T) == 4;
#pragma unroll
    for (int x = 0; x < NX; ++x) s[x] = (T)0;
    auto add = [&](T e, int c, bool on) {
#pragma clang fp contract(off)
      const T t0 = s[0] + e * w0[c];
      s[0] = on ? t0 : s[0];
      if constexpr (NX > 1) {
        const T t1 = s[1] + e * w1[c];
        s[1] = on ? t1 : s[1];
      }
    };
    if constexpr (F == RES_SHO) {
      // KW offsets in a few wide scalar loads: past the slice's list they are
      // the next slices' (or the padding's), inside the window all the same
      const int *__restrict__ t = a.tab + (p0 >> 6);
#pragma unroll
      for (int k = 0; k < KW; ++k) add(v[k], own + t[k], (m >> k) & 1u);
    } else if constexpr (!kF32) {
      constexpr int U = 8;
      const int b = sl < a.nslice ? a.tab[sl] - wb : 0;
      for (int k0 = 0; k0 < wd; k0 += U) {
        T v0[U], v1[U];
        unsigned cc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int idx = p0 + min(k0 + u, wd - 1) * 128 + 2 * lane;
          v0[u] = a.vals[idx];
          v1[u] = a.vals[idx + 1];
          cc[u] = *reinterpret_cast<const unsigned *>(a.c16 + idx);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          add(v0[u], b + (int)(cc[u] & 0xffffu), 2 * (k0 + u) < len);
          add(v1[u], b + (int)(cc[u] >> 16), 2 * (k0 + u) + 1 < len);
        }
      }
    } else {
      constexpr int U = 8;
      const int b = sl < a.nslice ? a.tab[sl] - wb : 0;
      for (int k0 = 0; k0 < wd; k0 += U) {
        T vv[U];
        int cc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int idx = p0 + min(k0 + u, wd - 1) * 64 + lane;
          vv[u] = a.vals[idx];
          cc[u] = b + (int)a.c16[idx];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) add(vv[u], cc[u], k0 + u < wd);
      }
    }
  }
};

// The workgroup's LDS beside the windows.
template <typename T>
struct ResShared {
  KStateT<T> st;
  // r and z of the vector step's partial sums (the first two), then
  // everyone's partial sums
  T part[3][kResRows];
  T wave[16 * 3];
  T tot[3][4];
  int fail;
};

// Sum over a 256-row group's rows of val, as the launched SpMV's workgroup
// publishes it (block_publish with 256 threads), for the workgroup's four
// groups; slot: this thread's, of `stride` to a value.
template <typename T, int NV>
__device__ __forceinline__ void publish_groups(int stride, ResShared<T> &sh, Word *w, unsigned e, int slot,
                                               const T (&val)[NV]) {
  const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const T s = row_wave_sum(val[k]);
    if (lane == 0) sh.wave[16 * k + wv] = s;
  }
  stores_done();  // the vector entries go before the partial sums
  __syncthreads();
  if (threadIdx.x < 4 * NV) {
    const int k = (int)threadIdx.x >> 2;
    if (slot >= 0) {
      T t = (T)0;
      for (int i = 0; i < 4; ++i) t += sh.wave[16 * k + 4 * ((int)threadIdx.x & 3) + i];
      publish(w + ((size_t)k * stride + slot) * kWords<T>, e, t);
    }
  }
}

// Partial sums of the vector step over this workgroup's four tiles of 256
// rows, a row of each to a thread (block_publish after CgTile::step, or after
// BiCGStab's vector steps); tile k begins at row first + k * apart.
template <typename T, int NV>
__device__ __forceinline__ void publish_rows(const ResArgs<T> &a, ResShared<T> &sh, Word *w, unsigned e, int first,
                                             int apart) {
  const int tid = (int)threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid < 256) {
    T acc[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = (T)0;
#pragma unroll
    for (int k = 0; k < kVI; ++k) {
      const int i = k * kVecBlock + tid;
      if (first + k * apart + tid < a.n) {
        const T ri = sh.part[0][i], zi = sh.part[1][i];
        acc[0] += ri * zi;
        if constexpr (NV > 1) acc[1] += ri * ri;
      }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const T s = row_wave_sum(acc[k]);
      if (lane == 0) sh.wave[16 * k + wv] = s;
    }
  }
  stores_done();  // the vector entries go before the partial sums
  __syncthreads();
  if (tid < NV) {
    T t = (T)0;
    for (int i = 0; i < 4; ++i) t += sh.wave[16 * tid + i];
    publish(w + ((size_t)tid * a.vec_grid + blockIdx.x) * kWords<T>, e, t);
  }
}

// Waits for everyone's partial sums, one workgroup's to a thread with all
// its words in flight, and adds them in block_reduce_all's order (256
// threads).  False: someone gave up.
template <typename T, int NV, bool SPMV>
__device__ __forceinline__ bool gather(const ResArgs<T> &a, ResShared<T> &sh, const Word *w, unsigned e, bool used,
                                       T (&tot)[NV]) {
  const int tid = (int)threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int g = SPMV ? a.spmv_grid : a.vec_grid;  // at most 1024
  T v[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = (T)0;
  if (used) {
    for (int spins = 0;; ++spins) {
      bool all = true;
#pragma unroll
      for (int k = 0; k < NV; ++k) all &= seen(w + ((size_t)k * g + tid) * kWords<T>, e, v[k]);
      if (all) break;
      if (spins > kSpins ||
          ((spins & 63) == 63 && __hip_atomic_load(a.gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        __hip_atomic_store(a.gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh.fail = 1;
        break;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) sh.part[k][tid] = v[k];
  __syncthreads();
  if (tid < 256) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      T s = (T)0;
#pragma unroll
      for (int u = 0; u < 4; ++u) s += sh.part[k][tid + 256 * u];
      s = row_wave_sum(s);
      if (lane == 0) sh.tot[k][wv] = s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    T t = (T)0;
    for (int i = 0; i < 4; ++i) t += sh.tot[k][i];
    tot[k] = t;
  }
  return sh.fail == 0;
}

// Calls f(c, entries of e0 (and e1) at column c) for the halo columns of
// each TH threads' rows, kHaloU columns of a thread in flight.
constexpr int kHaloU = 6;
template <typename T, int TH, int NE, class Fn>
__device__ __forceinline__ void halo_columns(int lo, int nlow, int re, int nhalo, const T *e0, const T *e1, Fn f) {
  for (int i0 = (int)threadIdx.x & (TH - 1); i0 < nhalo; i0 += kHaloU * TH) {
    T v[NE][kHaloU];
#pragma unroll
    for (int u = 0; u < kHaloU; ++u) {
      const int i = min(i0 + u * TH, nhalo - 1);
      const int c = i < nlow ? lo + i : re + (i - nlow);
      v[0][u] = ld_agent(e0 + c);
      if constexpr (NE > 1) v[1][u] = ld_agent(e1 + c);
    }
#pragma unroll
    for (int u = 0; u < kHaloU; ++u) {
      const int i = i0 + u * TH;
      if (i < nhalo) f(i < nlow ? lo + i : re + (i - nlow), v[0][u], v[NE - 1][u]);
    }
  }
}

}  // namespace

// One CG sequence, or `cap` iterations of it: it then stops between two, in
// the state of the launched loop there, and the next launch goes on.
// FAITHFUL: HUTI's order with the true residual of every
// iteration; its product A x and the next iteration's A p are taken in one
// pass over the matrix.  Else the one-SpMV order (FinCgFast2's tests).
template <typename T, ResFmt F, int KW, bool FAITHFUL>
__global__ __launch_bounds__(kResRows) void k_resident_cg(ResArgs<T> a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ ResShared<T> sh;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int R0 = (int)blockIdx.x * kResRows, r = R0 + tid, rl = min(r, a.n - 1);
  const bool ok = r < a.n;
  const int sl = __builtin_amdgcn_readfirstlane(R0 / 64 + (tid >> 6));
  const int wb = R0 - a.halo, own = tid + a.halo;  // the window's first column, this row's place
  const int lo = max(wb, 0), re = min(R0 + kResRows, a.n);  // the halo: [lo, R0) and [re, we)
  const int we = min(R0 + kResRows + a.halo, a.n);
  const int nlow = R0 - lo, nhalo = nlow + (we - re);
  T *win = reinterpret_cast<T *>(lds);     // z, or p with FAITHFUL
  T *winx = win + (kResRows + 2 * a.halo); // x (FAITHFUL)
  T x = a.v.x[rl], p = a.v.p[rl], q = a.v.q[rl], rr = a.v.r[rl], z = a.v.z[rl];
  const T dg = a.v.dg[rl];
  const T b = FAITHFUL ? a.v.b[rl] : (T)0, d = FAITHFUL && a.du ? a.du[rl] : (T)1;
  ResRow<T, F, KW> row;
  row.load(a, sl, lane);
  if (tid == 0) {
    sh.st = *a.st;
    sh.fail = 0;
  }
  {
    const T *src = FAITHFUL ? a.v.p : a.v.z;
    for (int i = tid; i < kResRows + 2 * a.halo; i += kResRows) {
      const int c = wb + i;
      win[i] = c >= 0 && c < a.n ? src[c] : (T)0;
      if constexpr (FAITHFUL) winx[i] = (T)0;
    }
  }
  __syncthreads();
  double *const hist = blockIdx.x == 0 ? a.hist : nullptr;
  const int slot = group_slot((int)blockIdx.x * 4 + (tid & 3), a.ngroups);
  const bool used = tid < a.spmv_grid && slot_used(tid, a.ngroups);
  unsigned e = 1;
  int left = a.cap;
  T sx[FAITHFUL ? 2 : 1];
  bool lost = false;
  if constexpr (FAITHFUL) {
    T s[1];
    row.template sums<1>(a, sl, lane, wb, own, win, win, s);
    q = s[0];
    T acc[3] = {(T)0, (T)0, (T)0};
    if (ok) acc[0] += p * q;
    publish_groups<T, 3>(a.spmv_grid, sh, a.w1, e, slot, acc);
  }
  if (!sh.st.done) for (bool first = true;; first = false) {
    T pq;
    if constexpr (FAITHFUL) {
      T tot[3];
      if (!gather<T, 3, true>(a, sh, a.w1, e, used, tot)) { lost = true; break; }
      if (!first) {
        T two[2] = {tot[1], tot[2]};
        EpiCgResidual<T> f{a.v, &sh.st, nullptr, 0, nullptr, hist, nullptr, 0, (T)0, a.du};
        f.finish(two);
        __syncthreads();
        if (sh.st.done || --left == 0) break;
      }
      pq = tot[0];
    } else {
      row.template sums<1>(a, sl, lane, wb, own, win, win, sx);
      const T beta = sh.st.beta;
      q = sx[0] + beta * q;
      p = z + beta * p;
      T acc[1] = {(T)0};
      if (ok) acc[0] += p * q;
      publish_groups<T, 1>(a.spmv_grid, sh, a.w1, e, slot, acc);
      T tot[1];
      if (!gather<T, 1, true>(a, sh, a.w1, e, used, tot)) { lost = true; break; }
      pq = tot[0];
    }
    ++e;
    const T alpha = sh.st.rho / pq;
    x = x + alpha * p;
    rr = rr - alpha * q;
    z = rr / dg;
    if (ok) {
      st_agent(a.ez + r, z);
      if constexpr (FAITHFUL) st_agent(a.ex + r, x);
    }
    sh.part[0][tid] = rr;
    sh.part[1][tid] = z;
    if (!FAITHFUL && ok) win[own] = z;
    __syncthreads();
    if constexpr (FAITHFUL) {
      publish_rows<T, 1>(a, sh, a.w2, e, R0, kVecBlock);
      T rn[1];
      if (!gather<T, 1, false>(a, sh, a.w2, e, tid < (int)gridDim.x, rn)) { lost = true; break; }
      const T beta = rn[0] / sh.st.rho;
      p = z + beta * p;
      halo_columns<T, kResRows, 2>(lo, nlow, re, nhalo, a.ez, a.ex, [&](int c, T zc, T xc) {
        win[c - wb] = zc + beta * win[c - wb];
        winx[c - wb] = xc;
      });
      if (ok) {
        win[own] = p;
        winx[own] = x;
      }
      __syncthreads();
      if (tid == 0) {
        sh.st.pq = pq;
        sh.st.alpha = alpha;
        sh.st.rho_new = rn[0];
      }
      row.template sums<2>(a, sl, lane, wb, own, win, winx, sx);
      q = sx[0];
      T acc[3] = {(T)0, (T)0, (T)0};
      if (ok) {
        acc[0] += p * q;
        const T ti = sx[1] - b;
        acc[1] += ti * ti;
        const T ui = ti / d;
        acc[2] += ui * ui;
      }
      ++e;
      publish_groups<T, 3>(a.spmv_grid, sh, a.w1, e, slot, acc);
    } else {
      publish_rows<T, 2>(a, sh, a.w2, e, R0, kVecBlock);
      T tot[2];
      if (!gather<T, 2, false>(a, sh, a.w2, e, tid < (int)gridDim.x, tot)) { lost = true; break; }
      if (tid == 0) {
        sh.st.pq = pq;
        sh.st.alpha = alpha;
      }
      FinCgFast2<T>{&sh.st, nullptr, 0, hist}.finish(tot);
      halo_columns<T, kResRows, 1>(lo, nlow, re, nhalo, a.ez, a.ez, [&](int c, T zc, T) { win[c - wb] = zc; });
      __syncthreads();
      if (sh.st.done || --left == 0) break;
      ++e;
    }
  }
  if (lost) return;  // nothing is committed
  if (ok) {
    a.out.x[r] = x;
    a.out.r[r] = rr;
    a.out.z[r] = z;
    a.out.p[r] = p;
    a.out.q[r] = q;
  }
  if (blockIdx.x == 0 && tid == 0) {
    sh.st.fresh = 1;
    *a.st_out = sh.st;
  }
}

// One BiCGStab sequence (or `cap` iterations) in huti_bicgstab.src order, four
// exchanges an iteration.  FAITHFUL: the true residual of every iteration, its product
// A x taken in one pass with the next iteration's A t1v; else FinBiXr's tests
// on the recurrence residual.  The halo's t1v = (r + beta w) / dg needs beta,
// so r and w = p - omega v travel with the partial sums that give it.
// A thread's tile of 256 rows is k of the workgroup's four, a whole number of
// grids apart; its window begins at k (256 + 2 halo).
template <typename T, ResFmt F, int KW, bool FAITHFUL>
__global__ __launch_bounds__(kResRows) void k_resident_bi(ResArgs<T> a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ ResShared<T> sh;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int k = __builtin_amdgcn_readfirstlane(tid >> 8), t = tid & (kVecBlock - 1);
  const int apart = (int)gridDim.x * kVecBlock, T0 = (int)blockIdx.x * kVecBlock;
  const int R0 = T0 + k * apart, r = R0 + t, rl = min(r, a.n - 1);
  const bool ok = r < a.n;
  const int sl = __builtin_amdgcn_readfirstlane(R0 / 64 + (t >> 6));
  const int width = kVecBlock + 2 * a.halo;
  const int wb = R0 - a.halo - k * width, own = k * width + t + a.halo;
  const int lo = max(R0 - a.halo, 0), re = min(R0 + kVecBlock, a.n);
  const int we = min(R0 + kVecBlock + a.halo, a.n);
  const int nlow = R0 - lo, nhalo = R0 < a.n ? nlow + (we - re) : 0;
  T *win = reinterpret_cast<T *>(lds);  // t1v and t2v in turn
  T *winx = win + 4 * width;            // x (FAITHFUL)
  T x = a.v.x[rl], p = a.v.p[rl], v = a.v.v[rl], rr = a.v.r[rl], t1 = a.v.t1v[rl];
  const T dg = a.v.dg[rl], rt = a.v.rtld[rl];
  const T b = FAITHFUL ? a.v.b[rl] : (T)0, d = FAITHFUL && a.du ? a.du[rl] : (T)1;
  ResRow<T, F, KW> row;
  row.load(a, sl, lane);
  if (tid == 0) {
    sh.st = *a.st;
    sh.fail = 0;
  }
  for (int i = k * width + t; i < (k + 1) * width; i += kVecBlock) {
    const int c = wb + i;
    win[i] = c >= 0 && c < a.n ? a.v.t1v[c] : (T)0;
    if constexpr (FAITHFUL) winx[i] = (T)0;
  }
  __syncthreads();
  double *const hist = blockIdx.x == 0 ? a.hist : nullptr;
  const int slot = group_slot((int)blockIdx.x + (tid & 3) * (int)gridDim.x, a.ngroups);
  const bool used = tid < a.spmv_grid && slot_used(tid, a.ngroups);
  unsigned e = 0;
  int left = a.cap;
  bool lost = false;
  if (!sh.st.done) for (bool first = true;; first = false) {
    ++e;
    if (FAITHFUL && !first) {
      T s[2];
      row.template sums<2>(a, sl, lane, wb, own, win, winx, s);
      v = s[0];
      T acc[3] = {(T)0, (T)0, (T)0};
      if (ok) {
        acc[0] += rt * v;
        const T ti = s[1] - b;
        acc[1] += ti * ti;
        const T ui = ti / d;
        acc[2] += ui * ui;
      }
      publish_groups<T, 3>(a.spmv_grid, sh, a.w1, e, slot, acc);
    } else {
      T s[1];
      row.template sums<1>(a, sl, lane, wb, own, win, win, s);
      v = s[0];
      T acc[3] = {(T)0, (T)0, (T)0};
      if (ok) acc[0] += rt * v;
      publish_groups<T, 3>(a.spmv_grid, sh, a.w1, e, slot, acc);
    }
    T rv[3];
    if (!gather<T, 3, true>(a, sh, a.w1, e, used, rv)) { lost = true; break; }
    if (FAITHFUL && !first) {
      T two[2] = {rv[1], rv[2]};
      EpiBiResidual<T> f{a.v, &sh.st, nullptr, 0, nullptr, hist, (T)0, (T)0, a.du};
      f.finish(two);
      __syncthreads();
      if (sh.st.done || --left == 0) break;
    }
    const T alpha = sh.st.rho / rv[0];
    const T s = rr - alpha * v;
    const T t2 = s / dg;
    if (ok) st_agent(a.ez + r, t2);
    if (ok) win[own] = t2;
    sh.part[0][tid] = s;
    sh.part[1][tid] = s;
    ++e;
    __syncthreads();
    publish_rows<T, 1>(a, sh, a.w2, e, T0, apart);
    T ss[1];
    if (!gather<T, 1, false>(a, sh, a.w2, e, tid < (int)gridDim.x, ss)) { lost = true; break; }
    if (tid == 0) sh.st.alpha = alpha;
    FinSnorm<T>{&sh.st, nullptr, 0}.finish(ss);
    halo_columns<T, kVecBlock, 1>(lo, nlow, re, nhalo, a.ez, a.ez, [&](int c, T tc, T) { win[c - wb] = tc; });
    __syncthreads();
    if (sh.st.snorm_exit) {
      x = x + alpha * t1;
      if (tid == 0) sh.st.done = 1;
      break;
    }
    T tv;
    {
      T q[1];
      row.template sums<1>(a, sl, lane, wb, own, win, win, q);
      tv = q[0];
    }
    {
      T acc[2] = {(T)0, (T)0};
      if (ok) {
        acc[0] += tv * s;
        acc[1] += tv * tv;
      }
      ++e;
      publish_groups<T, 2>(a.spmv_grid, sh, a.w1, e, slot, acc);
    }
    T tt[2];
    if (!gather<T, 2, true>(a, sh, a.w1, e, used, tt)) { lost = true; break; }
    const T omega = tt[0] / tt[1];
    x = x + alpha * t1 + omega * t2;
    rr = s - omega * tv;
    const T w = p - omega * v;
    if (ok) {
      st_agent(a.er + r, rr);
      st_agent(a.ew + r, w);
      if constexpr (FAITHFUL) st_agent(a.ex + r, x);
    }
    sh.part[0][tid] = rr;
    sh.part[1][tid] = rt;
    ++e;
    __syncthreads();
    publish_rows<T, 2>(a, sh, a.w2, e, T0, apart);
    T rn[2];
    if (!gather<T, 2, false>(a, sh, a.w2, e, tid < (int)gridDim.x, rn)) { lost = true; break; }
    if (tid == 0) {
      sh.st.ts = tt[0];
      sh.st.tt = tt[1];
      sh.st.omega = omega;
    }
    FinBiXr<T>{&sh.st, nullptr, 0, FAITHFUL ? 0 : 1, hist}.finish(rn);
    __syncthreads();
    if (!FAITHFUL && sh.st.done) break;
    const T beta = FAITHFUL ? (sh.st.rho_new * alpha) / (sh.st.rho * omega) : sh.st.beta;
    p = rr + beta * w;
    t1 = p / dg;
    halo_columns<T, kVecBlock, 2>(lo, nlow, re, nhalo, a.er, a.ew,
                       [&](int c, T rc, T wc) { win[c - wb] = (rc + beta * wc) / a.v.dg[c]; });
    if constexpr (FAITHFUL)
      halo_columns<T, kVecBlock, 1>(lo, nlow, re, nhalo, a.ex, a.ex, [&](int c, T xc, T) { winx[c - wb] = xc; });
    if (ok) {
      win[own] = t1;
      if constexpr (FAITHFUL) winx[own] = x;
    }
    __syncthreads();
    if (!FAITHFUL && --left == 0) break;
  }
  if (lost) return;  // nothing is committed
  if (ok) {
    a.out.x[r] = x;
    a.out.r[r] = rr;
    a.out.p[r] = p;
    a.out.v[r] = v;
    a.out.t1v[r] = t1;
  }
  __syncthreads();
  if (blockIdx.x == 0 && tid == 0) *a.st_out = sh.st;
}

template <typename T>
__global__ __launch_bounds__(256) void k_resident_commit(int n, Vecs<T> v, Vecs<T> out, KStateT<T> *st,
                                                         const KStateT<T> *st_out, const int *gave_up) {
  if (*gave_up) {
    if (blockIdx.x == 0 && threadIdx.x == 0) st->ticket[3] = 1;
    return;
  }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    v.x[i] = out.x[i];
    v.r[i] = out.r[i];
    v.p[i] = out.p[i];
    if (out.q) {  // CG
      v.z[i] = out.z[i];
      v.q[i] = out.q[i];
    } else {
      v.v[i] = out.v[i];
      v.t1v[i] = out.t1v[i];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *st = *st_out;
}

__global__ void k_resident_clear(Word *w, int nw, int *gave_up, unsigned *mark, int give_up) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nw; i += gridDim.x * blockDim.x) w[i] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *gave_up = give_up;
    *mark = 0;
  }
}

// One device, as this process's solves use it.
struct Device {
  std::mutex mu;
  int cus = 0;     // of the device; 0: not asked yet
  int solves = 0;  // solves, batches and servers with work in progress
  int launched = 0;  // those of them that launch their kernels
  int held = 0;    // CUs of an XCD that resident loops may hold
  std::chrono::steady_clock::time_point rest{};  // no resident loop before
};
static Device g_device[64];
static Device &device(const ehip_system *s) { return g_device[s->dev & 63]; }

// After a grid gave up, how long solves on the device stay launched.
constexpr std::chrono::seconds kRest(10);

// Workgroups go to the XCDs in turn, so a grid of g takes at most ceil(g / 8)
// CUs of any one of them.
static int cus_of_xcd(const Device &d, int g) {
  const int xcds = std::max(1, d.cus / kCusPerXcd);
  return (g + xcds - 1) / xcds;
}

DeviceUse::DeviceUse(int device, bool launched) : dev(device & 63), launched(launched) {
  std::lock_guard<std::mutex> lk(g_device[dev].mu);
  ++g_device[dev].solves;
  g_device[dev].launched += launched;
}
DeviceUse::~DeviceUse() {
  std::lock_guard<std::mutex> lk(g_device[dev].mu);
  --g_device[dev].solves;
  g_device[dev].launched -= launched;
}
void DeviceUse::launch() {
  std::lock_guard<std::mutex> lk(g_device[dev].mu);
  g_device[dev].launched += !launched;
  launched = true;
}

// Room for a resident loop of g workgroups.  Four host threads that solve
// together, resident loops one at a time / so / all launched, a round of four
// solves: 17^3 Hex8 in HUTI's order 2.9 / 2.7 / 3.8 ms, 47^3 12.2 / 9.9 / 10.7
// ms, 60^3 mixed 12.1 / 9.3 / 9.3 ms, 200^2 Quad4 BiCGStab 19.5 / 12.0 / 26.8 ms.
// One thread's launched work beside another's solves, resident / so / launched:
// an 80^3 mixed CG beside 301^2 BiCGStab 42 / 11.2 / 10.6 ms, a batch of five
// Quad4 systems beside 500^2 BiCGStab 260 / 11.5 / 12.1 ms.  A 17^3 solve beside
// 301^2 ones whose stream shares its hardware queue, in whole sequences / so /
// launched: 20 / 5.4 / 4.0 ms (1.0 on another queue, 1.9 launched).
bool resident_admit(const ehip_system *s, int g) {
  Device &d = device(s);
  std::lock_guard<std::mutex> lk(d.mu);
  if (!d.cus && hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, s->dev) != hipSuccess) {
    d.cus = 0;
    return false;
  }
  const int xcds = std::max(1, d.cus / kCusPerXcd), need = cus_of_xcd(d, g);
  if (d.launched > 0 || d.held + need > d.cus / xcds) return false;
  if (std::chrono::steady_clock::now() < d.rest) return false;
  d.held += need;
  return true;
}
void resident_release(const ehip_system *s, int g, bool gave_up) {
  Device &d = device(s);
  std::lock_guard<std::mutex> lk(d.mu);
  d.held -= cus_of_xcd(d, g);
  if (gave_up) d.rest = std::chrono::steady_clock::now() + kRest;
}

static int slice(const ehip_system *s) {
  if (s->resident_test == 3) return 1;
  Device &d = device(s);
  std::lock_guard<std::mutex> lk(d.mu);
  return d.solves > 1 ? kSliceShared : kSlice;
}

// CG: 1024 rows to a workgroup; BiCGStab: the launched vector steps' grid
int resident_groups(int n, bool cg) { return cg ? (n + kResRows - 1) / kResRows : vec_grid(n); }

// Words of the exchanges: three SpMV values of up to 1024 groups, two
// vector values of up to 1024 tiles, two words each.
constexpr int kW1 = 3 * 1024 * 2, kW2 = 2 * 1024 * 2;

// Values in a workgroup's window: its rows (BiCGStab: four tiles) and the
// halo on both sides.
static int64_t window(bool cg, int halo) {
  return cg ? kResRows + 2 * (int64_t)halo : 4 * (kVecBlock + 2 * (int64_t)halo);
}

// Rows per workgroup times CUs bound n; two windows must fit the LDS (one in
// the orders that test the recurrence residual).
template <typename T>
bool resident_fits(ehip_system *s, bool cg, bool faithful) {
  const int fmt = sizeof(T) == 4 ? s->fmt32 : s->fmt64;
  const int halo = fmt == 2 ? s->sho_halo : s->sell_halo;
  if (s->n > kResRows * kResGroups || halo < 0 || s->n < 1) return false;
  if (fmt == 2) {
    if (!s->sho_ok || s->sho_d != 1) return false;
  } else if (fmt == 1) {
    if (!s->sell_ok || s->sellb_d || s->sell_row || !s->sell_c16) return false;
    if (sizeof(T) == 8 && !s->sell2_ok) return false;
  } else {
    return false;
  }
  const int64_t win = window(cg, halo) * (int64_t)sizeof(T) * (faithful ? 2 : 1);
  return win + (int64_t)sizeof(ResShared<T>) + 64 <= kResLds;
}

static size_t vec_len(int n) { return ((size_t)n + 63) / 64 * 64; }

// The exchange words and vectors, allocated at first use.
bool resident_buffers(ehip_system *s) {
  const size_t need =
      (sizeof(Word) * (kW1 + kW2) + sizeof(KState) + 256) + 9 * vec_len(s->n) * sizeof(double);
  if (!s->res_buf && dmalloc(s, &s->res_buf, need)) return false;
  return true;
}

// Enqueues the sequence and its commit; the caller has the buffers and is
// admitted from here until it has read the state back, whose ticket[3] tells
// that the grid gave up and nothing changed.
template <typename T, bool CG>
static int resident_run(ehip_system *s, const Vecs<T> &v, KStateT<T> *st, bool faithful, double *hist, const T *du) {
  const int n = s->n;
  const size_t vec = vec_len(n);
  char *p = (char *)s->res_buf;
  ResArgs<T> a{};
  a.w1 = (Word *)p;
  a.w2 = a.w1 + kW1;
  p += sizeof(Word) * (kW1 + kW2);
  a.st_out = (KStateT<T> *)p;
  p += (sizeof(KState) + 63) / 64 * 64;
  a.gave_up = (int *)p;
  p += 64;
  T *w = (T *)p;
  a.ex = w;
  a.ez = w + vec;
  a.er = w + 2 * vec;
  a.ew = w + 3 * vec;
  a.out.x = w + 4 * vec;
  a.out.r = w + 5 * vec;
  a.out.p = w + 6 * vec;
  (CG ? a.out.z : a.out.v) = w + 7 * vec;
  (CG ? a.out.q : a.out.t1v) = w + 8 * vec;
  a.v = v;
  a.st = st;
  a.n = n;
  a.nslice = s->nslice;
  a.ngroups = (s->nslice + 3) / 4;
  a.spmv_grid = sell_grid(s);
  a.cap = slice(s);
  const int g = resident_groups(n, CG);
  a.vec_grid = CG ? fused_grid(n) : g;
  a.hist = hist;
  a.du = du;
  const int fmt = sizeof(T) == 4 ? s->fmt32 : s->fmt64;
  a.halo = fmt == 2 ? s->sho_halo : s->sell_halo;
  if (fmt == 2) {
    if constexpr (sizeof(T) == 4) a.vals = sho_values32(s); else a.vals = sho_values64(s);
    a.off = s->sho_off;
    a.tab = s->sho_tab;
    a.mask = s->sho_mask;
  } else {
    if constexpr (sizeof(T) == 4) {
      a.vals = sell_values32(s);
      a.off = s->sell_off;
      a.c16 = s->sell_c16;
    } else {
      a.vals = sell_values64(s);
      a.off = s->sell2_off;
      a.c16 = s->sell2_c16;
    }
    a.rows = s->rows;
    a.tab = s->sell_base;
  }
  if (!a.vals) return EHIP_ENOMEM;
  const size_t lds = (size_t)window(CG, a.halo) * sizeof(T) * (faithful ? 2 : 1);
  hipLaunchKernelGGL(k_resident_clear, dim3(16), dim3(256), 0, s->stream, a.w1, kW1 + kW2, a.gave_up, &st->ticket[3],
                     s->resident_test == 2 ? 1 : 0);
#define EHIP_RES(F, KW)                                                                                            \
  if constexpr (CG) {                                                                                              \
    if (faithful) hipLaunchKernelGGL((k_resident_cg<T, F, KW, true>), dim3(g), dim3(kResRows), lds, s->stream, a); \
    else hipLaunchKernelGGL((k_resident_cg<T, F, KW, false>), dim3(g), dim3(kResRows), lds, s->stream, a);         \
  } else {                                                                                                         \
    if (faithful) hipLaunchKernelGGL((k_resident_bi<T, F, KW, true>), dim3(g), dim3(kResRows), lds, s->stream, a); \
    else hipLaunchKernelGGL((k_resident_bi<T, F, KW, false>), dim3(g), dim3(kResRows), lds, s->stream, a);         \
  }
  // the widest slice's entries in registers: 9 (Quad4), 15 (Tet4), 27 (Hex8)
  if (fmt != 2) { EHIP_RES(RES_SELL, 1); }
  else if (s->sho_wmax <= 9) { EHIP_RES(RES_SHO, 9); }
  else if (s->sho_wmax <= 15) { EHIP_RES(RES_SHO, 15); }
  else if (s->sho_wmax <= 27) { EHIP_RES(RES_SHO, 27); }
  else { EHIP_RES(RES_SHO, 32); }
#undef EHIP_RES
  EHIP_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_resident_commit<T>, dim3(vec_grid(n)), dim3(256), 0, s->stream, n, v, a.out, st,
                     (const KStateT<T> *)a.st_out, (const int *)a.gave_up);
  EHIP_HIP_TRY(hipGetLastError());
  return EHIP_OK;
}

template <typename T>
int resident_cg(ehip_system *s, const Vecs<T> &v, KStateT<T> *st, bool faithful, double *hist, const T *du) {
  return resident_run<T, true>(s, v, st, faithful, hist, du);
}
template <typename T>
int resident_bicgstab(ehip_system *s, const Vecs<T> &v, KStateT<T> *st, bool faithful, double *hist, const T *du) {
  return resident_run<T, false>(s, v, st, faithful, hist, du);
}

// Tests: mode 0 as usual, 1 launched loops only, 2 every grid is told that a
// thread of its gave up (it ends as ever and commits nothing), 3 launches of
// one iteration each.  Ends the device's rest.
extern "C" int ehip_internal_resident(ehip_system *s, int mode) {
  if (!s) return EHIP_EARG;
  s->resident_test = mode;
  Device &d = device(s);
  std::lock_guard<std::mutex> lk(d.mu);
  d.rest = {};
  return EHIP_OK;
}

template bool resident_fits<double>(ehip_system *, bool, bool);
template bool resident_fits<float>(ehip_system *, bool, bool);
template int resident_cg<double>(ehip_system *, const Vecs<double> &, KStateT<double> *, bool, double *,
                                 const double *);
template int resident_cg<float>(ehip_system *, const Vecs<float> &, KStateT<float> *, bool, double *, const float *);
template int resident_bicgstab<double>(ehip_system *, const Vecs<double> &, KStateT<double> *, bool, double *,
                                       const double *);
template int resident_bicgstab<float>(ehip_system *, const Vecs<float> &, KStateT<float> *, bool, double *,
                                      const float *);

}  // namespace ehip
