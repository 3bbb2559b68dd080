// hb_mixed.hip - mixed-precision CG with reliable updates.
//
// The inner iteration is the reference's CG (cg.F90:93-117) on the operator
// built from FP32 or 16-bit copies of the links and clover term, with FP32
// arithmetic and the search direction, residual and operator temporaries in
// the same storage precision (16-bit spinors carry a per-site FP32 scale).  The
// dot products accumulate in FP64.  A reliable update (defect correction)
// folds the low-precision solution increment into the FP64 solution and
// replaces the iterated residual by the FP64 true residual b - A x whenever the
// iterated residual has dropped by `delta` against its maximum since the last
// update, after `max_inner` iterations, or when it reaches the stopping bound.
// The solve stops only on the FP64 true residual (|r|^2 <= rest).
#include <cmath>

#include "hb_ops.h"

namespace hb {

// The scalars of an iteration, in two slots as those of the FP64 CG (CgState).
struct MixSlot {
  double rtr, maxr;  // iterated |r|^2; largest |r| since the last reliable update
  int iter, since;
  int flag;          // 0 iterate, 1 reliable update due, 2 converged, 3 maxiter reached
};
struct MixState {
  MixSlot s[2];
  double pap;           // <p, A p> of the iteration, from the r update for the p update
  double alpha[4];      // of the iterations whose x_lo updates are pending (MixRing)
  double beta;          // of the p update or of the restart after a reliable update
  int go;               // the iteration ran: its p update is due
  int cur;              // slot of the ring that holds the search direction at a reliable update
  double rp_re, rp_im;  // <r, p> / |r|^2 after a reliable update
  double rest, delta;
  int max_inner, maxiter;
  int n_reliable;
  double res[4];
};

// ---- precision conversion ----------------------------------------------------
template <class S>
__global__ void k_cvt_field(typename S::ST *__restrict__ dst, const double2 *__restrict__ src, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t k = i; k < n; k += (size_t)gridDim.x * blockDim.x) {
    double2 v = src[k];
    S::st(dst, k, cmk<typename S::V>((typename S::A)v.x, (typename S::A)v.y));
  }
}

// links in reduced precision, rows 0 and 1 only (U[4][2][6][vh], see load_link)
template <class S>
__global__ void k_cvt_gauge_rows(typename S::ST *__restrict__ dst, const double2 *__restrict__ src, size_t vh) {
  const size_t n = 48 * vh;
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x) {
    const size_t slab = k / (6 * vh), rem = k - slab * 6 * vh;
    const double2 v = src[slab * 9 * vh + rem];
    S::st(dst, k, cmk<typename S::V>((typename S::A)v.x, (typename S::A)v.y));
  }
}

// links in 16 bits: rows 0 and 1, a 16-byte and an 8-byte plane per (mu, eo)
// slab (see load_link_f)
__global__ void k_cvt_gauge16(short2 *__restrict__ dst, const double2 *__restrict__ src, int vh) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int slab = blockIdx.y;  // mu*2 + eo
  if (i >= vh) return;
  link_to_rec16(dst + (size_t)slab * 6 * vh, i, vh, src + (size_t)slab * 9 * vh + i, vh);
}

// clover in 16-bit storage: per site and block, c 1 + m Q (see clover_block_scale)
// in five 16-byte planes per [eo][J] slab (see load_clover_block_raw)
__global__ void k_cvt_clover16(short2 *__restrict__ dst, const double2 *__restrict__ src, int vh) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int eb = blockIdx.y;  // eo*2 + J
  if (i >= vh) return;
  clover_to_rec16(dst + (size_t)eb * kClov16Words * vh, i, vh, src + (size_t)eb * 18 * vh + i, vh);
}

// spinor FP64 -> S (thread per site: FP16 needs the site's norm)
template <class S>
__global__ void k_cvt_spinor(SpinorPtr<S> dst, const double2 *__restrict__ src, int vh) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  double2 v[12];
#pragma unroll
  for (int k = 0; k < 12; k++) v[k] = src[(size_t)k * vh + i];
  store_spinor<S>(dst, i, vh, v);
}

// reduced-precision field back to an FP64 spinor (the stored values, decoded)
template <class S>
__global__ void k_spinor_to_f64(double2 *__restrict__ dst, SpinorPtr<S> src, int vh) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  typename S::V v[12];
  load_spinor<S>(v, src, i, vh);
#pragma unroll
  for (int k = 0; k < 12; k++) dst[(size_t)k * vh + i] = make_double2((double)v[k].x, (double)v[k].y);
}

// ---- inner iteration kernels -----------------------------------------------------
// The solution increment since the last reliable update, x_lo, is FP32 (in 16
// bits its rounding, amplified by the operator's high modes, stalled the FP32
// inner solver).  The update x_lo += alpha p happens in the p update, which
// reads p anyway.

//
// Fields without a scale per site are updated one complex number per thread,
// 16-bit fields one site per thread; n counts what a thread works on.
template <class S> constexpr bool kLinear = !S::kNorm;
template <class S> inline int mix_count(int vh) { return kLinear<S> ? 12 * vh : vh; }
// 16-bit site kernels in workgroups of 64 / 256 sites, us per iteration: 2 k sites per
// parity 35.1 / 35.6, 21 k 42.8 / 43.6, 50 k 57.7 / 57.4, 74 k 76.0 / 74.3, 104 k 94.7 / 92.0
template <class S> inline int mix_block(int vh) { return !kLinear<S> && vh <= (1 << 16) ? 64 : kBlock; }
// (linear fields in at most 2048 blocks that go round; at most 1024 / 2048 / 4096, us
// per iteration: FP32 66 k 81.2 / 81.6 / 87.8, 200 k 218 / 220 / 228; FP64, which has the
// same cap, 104 k 178 / 178 / 187, 332 k 578 / 578 / 581)
template <class S> inline int mix_grid(int vh) {
  const int b = nblocks(mix_count<S>(vh), mix_block<S>(vh));
  return kLinear<S> && b > 2048 ? 2048 : b;
}

// The blocks sum the partials of a reduction themselves while their first
// operands are on their way (SUM), except in the site kernels of large
// lattices, which hold a whole site's operands in registers meanwhile and wait
// at the barrier: 16-bit updates at 32^3x64 74 us, with a finalize launch for
// each sum 64 + 8 us; at 12^3x24 7.2 against 6.3 + 5 us.  us per iteration, with the
// ring below in place of SUM / SUM: 104 k 96.1 / 92.2, 174 k 133 / 131, 249 k 170 / 171,
// 332 k 227 / 228, 432 k 296 / 299.
template <class S> inline bool mix_sum(int vh) { return kLinear<S> || vh <= (1 << 18); }
template <bool SUM> __device__ __forceinline__ double mix_total(const double *p, int n) {
  if constexpr (SUM) return partials_total(p, n);
  else return *p;
}

// what a thread works on: one number, or a site's twelve
template <class S> constexpr int kNums = kLinear<S> ? 1 : 12;
template <class S>
__device__ __forceinline__ void load_nums(typename S::V (&v)[kNums<S>], const SpinorPtr<S> &f, int i, int n) {
  if constexpr (kLinear<S>) v[0] = S::ld(f.p, i);
  else load_spinor<S>(v, f, i, n);
}
template <class S>
__device__ __forceinline__ void store_nums(const SpinorPtr<S> &f, int i, int n, const typename S::V (&v)[kNums<S>]) {
  if constexpr (kLinear<S>) S::st(f.p, i, v[0]);
  else store_spinor<S>(f, i, n, v);
}

// alpha = rtr / pAp; r -= alpha q; partial sums of |r|^2
template <class S, bool SUM>
__global__ __launch_bounds__(kBlock) void k_mix_update(SpinorPtr<S> r, SpinorPtr<S> q, int n, MixState *st, int k,
                                                       const double *pa, int na, double *pb) {
  using V = typename S::V;
  const MixSlot c = st->s[k & 1];
  if (c.flag) return;
  // the first operands are on their way while the partials are summed
  const int step = gridDim.x * blockDim.x;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  V qv[kNums<S>], rv[kNums<S>];
  if (SUM && i < n) {
    load_nums<S>(qv, q, i, n);
    load_nums<S>(rv, r, i, n);
    asm volatile("" ::: "memory");
  }
  const double pap = mix_total<SUM>(pa, na);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->pap = pap;
  const float alpha = (float)(c.rtr / pap);
  double s = 0.0;
  if (!SUM && i < n) {
    load_nums<S>(qv, q, i, n);
    load_nums<S>(rv, r, i, n);
  }
  while (i < n) {
    V v[kNums<S>];
#pragma unroll
    for (int m = 0; m < kNums<S>; m++) {
      v[m].x = rv[m].x - alpha * qv[m].x;
      v[m].y = rv[m].y - alpha * qv[m].y;
      s += (double)v[m].x * v[m].x + (double)v[m].y * v[m].y;
    }
    const int j = i + step;
    if (kLinear<S> && j < n) {
      load_nums<S>(qv, q, j, n);
      load_nums<S>(rv, r, j, n);
    }
    store_nums<S>(r, i, n, v);
    i = kLinear<S> ? j : n;
  }
  double vals[1] = {s};
  block_partials<1>(vals, pb);
}

// iterated |r|^2 -> reliable-update decision or beta (cg.F90:109-115): the slot
// of the next iteration; returns whether it goes on
__device__ __forceinline__ bool mix_decide(MixSlot &d, const MixSlot &c, const MixState *st, double rn) {
  const double rnorm = sqrt(rn);
  d = c;
  d.iter += 1;
  d.since += 1;
  if (rnorm > d.maxr) d.maxr = rnorm;
  const bool next = !(rn <= st->rest || rnorm < st->delta * d.maxr || d.since >= st->max_inner || d.iter >= st->maxiter);
  if (next) d.rtr = rn;
  else d.flag = 1;
  return next;
}

// small lattices: x_lo += alpha p, then p = r + beta p (unless a reliable
// update or the end is due)
template <class S>
__global__ __launch_bounds__(kBlock) void k_mix_pupdate(SpinorPtr<S> p, SpinorPtr<S> r, float2 *__restrict__ xlo, int n,
                                                        MixState *st, int k, const double *pb, int nb, Note note) {
  using V = typename S::V;
  const MixSlot c = st->s[k & 1];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (c.flag) {
    if (first) {
      st->s[~k & 1] = c;
      note.tell(c.flag);
    }
    return;
  }
  const int step = gridDim.x * blockDim.x;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  V pv[kNums<S>], rv[kNums<S>];
  float2 xv[kNums<S>];
  const auto load = [&](int j) {
    load_nums<S>(pv, p, j, n);
    load_nums<S>(rv, r, j, n);
#pragma unroll
    for (int m = 0; m < kNums<S>; m++) xv[m] = xlo[(size_t)m * n + j];
  };
  if (i < n) load(i);
  asm volatile("" ::: "memory");
  const double rn = partials_total(pb, nb);
  MixSlot d;
  const bool next = mix_decide(d, c, st, rn);
  const float alpha = (float)(c.rtr / st->pap);
  const float beta = (float)(rn / c.rtr);
  if (first) {
    st->s[~k & 1] = d;
    note.tell(d.flag);
  }
  while (i < n) {
    V v[kNums<S>];
#pragma unroll
    for (int m = 0; m < kNums<S>; m++) {
      xlo[(size_t)m * n + i] = make_float2(xv[m].x + alpha * pv[m].x, xv[m].y + alpha * pv[m].y);
      v[m].x = rv[m].x + beta * pv[m].x;
      v[m].y = rv[m].y + beta * pv[m].y;
    }
    if (next) store_nums<S>(p, i, n, v);
    i = kLinear<S> ? i + step : n;
    if (kLinear<S> && i < n) load(i);
  }
}

// Large lattices are bound by the bytes of the vector updates, half of them
// x_lo's.  Their search directions go round four buffers, p of iteration k in
// slot k & 3, and x_lo takes up four of them at a time (or those there are,
// when a reliable update is due): the same sums in the same order.  16-bit
// storage at 32^3x64: 34.9 us a launch against 43.0, an iteration 474 against 493.
// Without memory for three of the buffers (last = 0: the only slot of the ring)
// x_lo takes up every direction as it comes.
template <class S> struct MixRing {
  SpinorPtr<S> p[4];
};
struct FinMixStep {
  MixState *st;
  int k, last;
  Note note;
  __device__ void operator()(const double (&t)[1]) const {
    const MixSlot c = st->s[k & 1];
    MixSlot d = c;
    st->go = c.flag == 0;
    if (c.flag == 0) {
      mix_decide(d, c, st, t[0]);
      st->alpha[k & last] = c.rtr / st->pap;
      st->beta = t[0] / c.rtr;
      st->cur = k & last;
    }
    st->s[~k & 1] = d;
    note.tell(d.flag);
  }
};
template <class S>
__global__ __launch_bounds__(kBlock) void k_mix_pupdate_ring(MixRing<S> ring, SpinorPtr<S> r, float2 *__restrict__ xlo,
                                                             int n, const MixState *st, int k, int last) {
  using V = typename S::V;
  if (!st->go) return;
  const bool next = st->s[~k & 1].flag == 0;
  const int slot = k & last;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  V pv[12];
  if (slot == last || !next) {
    float2 x[12];
#pragma unroll
    for (int m = 0; m < 12; m++) x[m] = xlo[(size_t)m * n + i];
    for (int q = 0; q <= slot; q++) {
      const float alpha = (float)st->alpha[q];
      load_spinor<S>(pv, ring.p[q], i, n);
#pragma unroll
      for (int m = 0; m < 12; m++) {
        x[m].x += alpha * pv[m].x;
        x[m].y += alpha * pv[m].y;
      }
    }
#pragma unroll
    for (int m = 0; m < 12; m++) xlo[(size_t)m * n + i] = x[m];
  } else {
    load_spinor<S>(pv, ring.p[slot], i, n);
  }
  if (!next) return;
  const float beta = (float)st->beta;
  V rv[12];
  load_spinor<S>(rv, r, i, n);
#pragma unroll
  for (int m = 0; m < 12; m++) {
    pv[m].x = rv[m].x + beta * pv[m].x;
    pv[m].y = rv[m].y + beta * pv[m].y;
  }
  store_spinor<S>(ring.p[(k + 1) & last], i, n, pv);
}

// ---- reliable update kernels ------------------------------------------------------
// x += x_lo; x_lo = 0
__global__ void k_mix_accum(double2 *__restrict__ x, float2 *__restrict__ xlo, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t k = i; k < n; k += (size_t)gridDim.x * blockDim.x) {
    float2 d = xlo[k];
    double2 v = x[k];
    x[k] = make_double2(v.x + (double)d.x, v.y + (double)d.y);
    xlo[k] = make_float2(0.f, 0.f);
  }
}

// r = b - Ax (in place in ax), |r|^2; then r_lo = r and the scalar bookkeeping
template <class S>
__global__ __launch_bounds__(kBlock) void k_mix_true_residual(double2 *__restrict__ ax,
                                                              const double2 *__restrict__ b,
                                                              SpinorPtr<S> rlo, int vh,
                                                              double *partials) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0.0;
  if (i < vh) {
    double2 v[12];
#pragma unroll
    for (int k = 0; k < 12; k++) {
      double2 bb = b[(size_t)k * vh + i], a = ax[(size_t)k * vh + i];
      v[k] = make_double2(bb.x - a.x, bb.y - a.y);
      ax[(size_t)k * vh + i] = v[k];
      s += v[k].x * v[k].x + v[k].y * v[k].y;
    }
    store_spinor<S>(rlo, i, vh, v);
  }
  double vals[1] = {s};
  block_partials<1>(vals, partials);
}

// true |r|^2 -> convergence, or restart of the inner iteration
struct FinMixTrue {
  MixState *st;
  int first;
  Note note;
  __device__ void operator()(const double (&t)[1]) const {
    const double rt = t[0];
    MixSlot &c = st->s[0];
    st->res[0] = rt;
    if (!first) st->n_reliable += 1;
    c.since = 0;
    c.maxr = sqrt(rt);
    if (rt <= st->rest) {
      c.flag = 2;
    } else if (c.iter >= st->maxiter) {
      c.flag = 3;
    } else {
      // the true residual replaces the iterated one; the search direction is kept
      st->beta = first ? 0.0 : rt / c.rtr;
      c.rtr = rt;
      c.flag = 0;
    }
    note.tell(c.flag);
  }
};

// Re-orthogonalisation of the kept search direction at a reliable update:
// <r_lo, p> (complex) over the new residual, so that the restart can take out
// the component of p along r that the replaced residual no longer cancels
// (the reliable-update CG of Clark et al., "Solving lattice QCD systems of
// equations using mixed precision solvers on GPUs", 2010)
#ifndef HB_MIX_REORTH
#define HB_MIX_REORTH 1
#endif
template <class S>
__global__ __launch_bounds__(kBlock) void k_mix_rdotp(MixRing<S> ring, SpinorPtr<S> r, int vh, const MixState *st,
                                                      double *partials) {
  using V = typename S::V;
  if (st->s[0].flag) return;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double re = 0.0, im = 0.0;
  if (i < vh) {
    V pv[12], rv[12];
    load_spinor<S>(pv, ring.p[st->cur], i, vh);
    load_spinor<S>(rv, r, i, vh);
#pragma unroll
    for (int k = 0; k < 12; k++) {  // conj(r) p
      re += (double)rv[k].x * pv[k].x + (double)rv[k].y * pv[k].y;
      im += (double)rv[k].x * pv[k].y - (double)rv[k].y * pv[k].x;
    }
  }
  double vals[2] = {re, im};
  block_partials<2>(vals, partials);
}

struct FinMixRdotp {
  MixState *st;
  __device__ void operator()(const double (&t)[2]) const {
    st->rp_re = t[0] / st->s[0].rtr;
    st->rp_im = t[1] / st->s[0].rtr;
  }
};

// p = r_lo + beta (p - rp r_lo) after a reliable update (rp = <r, p>/|r|^2, or
// 0; beta = 0 at the start: p = r)
template <class S>
__global__ __launch_bounds__(kBlock) void k_mix_prestart(MixRing<S> ring, SpinorPtr<S> r, int vh,
                                                         const MixState *st) {
  using V = typename S::V;
  if (st->s[0].flag) return;
  const float beta = (float)st->beta;
  const float cr = (float)st->rp_re, ci = (float)st->rp_im;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  V pv[12], rv[12];
  load_spinor<S>(rv, r, i, vh);
  if (beta != 0.f) {
    load_spinor<S>(pv, ring.p[st->cur], i, vh);
  } else {
#pragma unroll
    for (int k = 0; k < 12; k++) pv[k] = cmk<V>(0.f, 0.f);
  }
#pragma unroll
  for (int k = 0; k < 12; k++) {
    const float ux = pv[k].x - (cr * rv[k].x - ci * rv[k].y);
    const float uy = pv[k].y - (cr * rv[k].y + ci * rv[k].x);
    pv[k].x = rv[k].x + beta * ux;
    pv[k].y = rv[k].y + beta * uy;
  }
  store_spinor<S>(ring.p[0], i, vh, pv);
}

// ---- low-precision copies of links and clover ------------------------------------
template <class S> struct LP;
template <> struct LP<SF32> {
  static const float2 *gauge(Context *c) { return c->gauge32; }
  static const float2 *clov(Context *c, int k) { return c->clov32[k]; }
  static const float *norm(Context *, int) { return nullptr; }
};
template <> struct LP<SF16> {
  static const short2 *gauge(Context *c) { return c->gauge16; }
  static const short2 *clov(Context *c, int k) { return c->clov16[k]; }
  static const float *norm(Context *, int) { return nullptr; }  // factors stored with the words
};

int ensure_lowprec(Context *c, int prec) {
  const size_t vh = c->g.vh;
  const bool clov = use_clover(c);
  if (c->lp_gauge_version == c->gauge_version * 1000 + prec &&
      c->lp_clover_version == c->clover_version * 1000 + prec)
    return HB_OK;
  const int grid = nblocks((int)std::min<size_t>(72 * vh, (size_t)1 << 22));
  if (prec == 32) {
    if (!c->gauge32) HB_HIP(device_alloc(c, &c->gauge32, sizeof(float2) * 48 * vh));
    k_cvt_gauge_rows<SF32><<<grid, kBlock, 0, c->stream>>>(c->gauge32, c->gauge, vh);
    HB_HIP(hipGetLastError());
    if (clov) {
      for (int k = 0; k < 2; k++) {
        if (!c->clov32[k]) HB_HIP(device_alloc(c, &c->clov32[k], sizeof(float2) * 72 * vh));
        k_cvt_field<SF32><<<grid, kBlock, 0, c->stream>>>(c->clov32[k], c->clov[k], 72 * vh);
        HB_HIP(hipGetLastError());
      }
    }
  } else {
    if (!c->gauge16) HB_HIP(device_alloc(c, &c->gauge16, sizeof(short2) * 48 * vh));
    k_cvt_gauge16<<<dim3(nblocks((int)vh), 8), kBlock, 0, c->stream>>>(c->gauge16, c->gauge, (int)vh);
    HB_HIP(hipGetLastError());
    if (clov) {
      for (int k = 0; k < 2; k++) {
        if (!c->clov16[k]) HB_HIP(device_alloc(c, &c->clov16[k], sizeof(short2) * 4 * kClov16Words * vh));
        k_cvt_clover16<<<dim3(nblocks((int)vh), 4), kBlock, 0, c->stream>>>(c->clov16[k], c->clov[k], (int)vh);
        HB_HIP(hipGetLastError());
      }
    }
  }
  c->lp_gauge_version = c->gauge_version * 1000 + prec;
  c->lp_clover_version = c->clover_version * 1000 + prec;
  return HB_OK;
}

// half of M~ (or M~^+) with spinors in S and links/clover in G; see mtil_f64
template <class S, class G>
int mtil_lp(Context *c, bool dag, double kappa, double rho, SpinorPtr<S> out, SpinorPtr<S> in,
            SpinorPtr<S> t, double *dot, SpinorPtr<S> dotv, const int *skip) {
  const bool clov = use_clover(c);
  DslashArgs<S, G> a1{};
  a1.g = c->g;
  a1.out_parity = 1;
  a1.out = t;
  a1.in = in;
  a1.U = LP<G>::gauge(c);
  a1.C = clov ? LP<G>::clov(c, HB_CLOVER_AINV) : nullptr;
  a1.Cn = clov ? LP<G>::norm(c, HB_CLOVER_AINV) : nullptr;
  a1.skip = skip;
  HB_TRY(launch_dslash(a1, dag, EPI_CLINV, c->stream));
  DslashArgs<S, G> a2{};
  a2.g = c->g;
  a2.out_parity = 0;
  a2.out = out;
  a2.in = t;
  a2.U = LP<G>::gauge(c);
  a2.C = clov ? LP<G>::clov(c, HB_CLOVER_A) : nullptr;
  a2.Cn = clov ? LP<G>::norm(c, HB_CLOVER_A) : nullptr;
  a2.x0 = in;
  a2.mkappa2 = -kappa * kappa;
  a2.rho = rho;
  a2.skip = skip;
  if (dot) {
    a2.dotv = dotv;
    a2.partials = dot;
    HB_TRY(launch_dslash(a2, dag, EPI_MTDOT, c->stream));
  } else {
    HB_TRY(launch_dslash(a2, dag, EPI_MTIL, c->stream));
  }
  return HB_OK;
}

template <class S> struct SpinorAlloc {
  static SpinorPtr<S> get(Context *c, int slot, int nslot, int *rc) {
    size_t vh = c->g.vh;
    size_t bytes = sizeof(typename S::ST) * 12 * vh;
    SpinorPtr<S> p{static_cast<typename S::ST *>(scratch(c, slot, bytes, rc)), nullptr};
    if (*rc) return p;
    if (S::kNorm) p.norm = static_cast<float *>(scratch(c, nslot, sizeof(float) * vh, rc));
    return p;
  }
};

template <class S, class G>
int cg_mixed_impl(Context *c, int op, double kappa, double rho, double2 *x, const double2 *b,
                  float rest, int maxiter, int log, double delta, int max_inner, int *iters,
                  int *n_rel, double *true_rtr) {
  const int vh = c->g.vh;
  const double r_op = op == HB_OP_WDAGW ? rho : 0.0;
  int rc = 0;
  // FP64 work fields
  double2 *t64 = spinor_scratch(c, SLOT_T, &rc); HB_TRY(rc);
  double2 *y64 = spinor_scratch(c, SLOT_Y, &rc); HB_TRY(rc);
  double2 *ax = spinor_scratch(c, SLOT_MIX0, &rc); HB_TRY(rc);
  float2 *xlo = static_cast<float2 *>(scratch(c, SLOT_MIX1, sizeof(float2) * 12 * (size_t)vh, &rc)); HB_TRY(rc);
  // low-precision fields (norm slots follow SLOT_LPN)
  SpinorPtr<S> p = SpinorAlloc<S>::get(c, SLOT_LP0, SLOT_LPN, &rc); HB_TRY(rc);
  const bool sums = mix_sum<S>(vh);
  SpinorPtr<S> r = SpinorAlloc<S>::get(c, SLOT_LP1, SLOT_LPN1, &rc); HB_TRY(rc);
  SpinorPtr<S> q = SpinorAlloc<S>::get(c, SLOT_LP2, SLOT_LPN2, &rc); HB_TRY(rc);
  SpinorPtr<S> t = SpinorAlloc<S>::get(c, SLOT_LP3, SLOT_LPN3, &rc); HB_TRY(rc);
  SpinorPtr<S> y = SpinorAlloc<S>::get(c, SLOT_LP4, SLOT_LPN4, &rc); HB_TRY(rc);
  MixState *st = static_cast<MixState *>(scratch(c, SLOT_STATE, sizeof(MixState), &rc)); HB_TRY(rc);
  HB_TRY(ensure_host_stage(c, sizeof(MixState)));
  MixState *hs = static_cast<MixState *>(c->host_stage);
  HB_TRY(ensure_lowprec(c, G::kBytes == 8 ? 32 : 16));
  MixRing<S> ring{{p, p, p, p}};
  const int last = !sums && spare_fields<S>(c, &ring.p[1], vh) ? 3 : 0;  // slot of the ring

  EventTimer tm;
  HB_TRY(tm.create());
  HB_TRY(tm.start(c->stream));
  MixState init{};
  init.rest = (double)rest;
  init.delta = delta;
  init.max_inner = max_inner;
  init.maxiter = maxiter;
  *hs = init;
  HB_HIP(hipMemcpyAsync(st, hs, sizeof(MixState), hipMemcpyHostToDevice, c->stream));
  HB_TRY(zero_f64(c, reinterpret_cast<double2 *>(xlo), (size_t)6 * vh));

  int nmv = 0;
  auto reliable = [&](int first) -> int {
    if (!first) {
      k_mix_accum<<<nblocks(std::min(12 * vh, 1 << 22)), kBlock, 0, c->stream>>>(x, xlo, (size_t)12 * vh);
      HB_HIP(hipGetLastError());
    }
    HB_TRY(apply_f64(c, op, kappa, rho, ax, x, t64, y64, nullptr, nullptr));
    k_mix_true_residual<S><<<nblocks(vh), kBlock, 0, c->stream>>>(ax, b, r, vh, c->red);
    k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(c->red, nblocks(vh), nullptr, FinMixTrue{st, first, next_note(c)});
    HB_HIP(hipGetLastError());
    if (!first && HB_MIX_REORTH) {
      k_mix_rdotp<S><<<nblocks(vh), kBlock, 0, c->stream>>>(ring, r, vh, st, c->red);
      k_finalize<2><<<1, kFinThreads, 0, c->stream>>>(c->red, nblocks(vh), &st->s[0].flag, FinMixRdotp{st});
      HB_HIP(hipGetLastError());
    }
    k_mix_prestart<S><<<nblocks(vh), kBlock, 0, c->stream>>>(ring, r, vh, st);
    HB_HIP(hipGetLastError());
    nmv++;
    return HB_OK;
  };
  HB_TRY(reliable(1));
  // partials of <p, A p> and of |r|^2
  const int na = dslash_grid<S, G>(vh), n = mix_count<S>(vh), grid = mix_grid<S>(vh), block = mix_block<S>(vh);
  double *pa = c->red, *pb = c->red + na + 1;
  Watch watch(c);
  for (int k = 0, flag = 0;;) {
    const int *skip = &st->s[k & 1].flag;
    const SpinorPtr<S> pk = ring.p[k & last];
    HB_TRY((mtil_lp<S, G>(c, false, kappa, r_op, y, pk, t, nullptr, SpinorPtr<S>{}, skip)));
    HB_TRY((mtil_lp<S, G>(c, true, kappa, r_op, q, y, t, pa, pk, skip)));
    const double *sum = pa;
    int nsum = na;
    HB_TRY(shorten_partials(c, sum, nsum, skip, sums ? kMaxParts : 1));
    const Note note = next_note(c);
    if (sums) {
      k_mix_update<S, true><<<grid, block, 0, c->stream>>>(r, q, n, st, k, sum, nsum, pb);
      k_mix_pupdate<S><<<grid, block, 0, c->stream>>>(p, r, xlo, n, st, k, pb, grid, note);
    } else if constexpr (!kLinear<S>) {
      k_mix_update<S, false><<<grid, block, 0, c->stream>>>(r, q, n, st, k, sum, nsum, pb);
      k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(pb, grid, nullptr, FinMixStep{st, k, last, note});
      k_mix_pupdate_ring<S><<<grid, block, 0, c->stream>>>(ring, r, xlo, n, st, k, last);
    }
    HB_HIP(hipGetLastError());
    HB_TRY(watch.look(&flag));
    k++;
    if (flag > 1) break;
    if (flag == 1) {
      HB_TRY(reliable(0));
      k = 0;  // goes on from slot 0 with the direction the restart left there
    }
  }
  HB_HIP(hipMemcpyAsync(hs, st, sizeof(MixState), hipMemcpyDeviceToHost, c->stream));
  HB_HIP(hipStreamSynchronize(c->stream));
  HB_TRY(tm.stop(c->stream));
  float ms = 0.f;
  HB_TRY(tm.elapsed(&ms));
  c->last_solve_ms = ms;
  c->last_n_matvec = nmv + hs->s[0].iter;
  if (iters) *iters = hs->s[0].iter;
  if (n_rel) *n_rel = hs->n_reliable;
  if (true_rtr) *true_rtr = hs->res[0];
  if (hs->s[0].flag != 2 && log != 2) {
    set_error("cg_mixed(): no convergence; true rtr = %.17g", hs->res[0]);
    return HB_E_NOCONV;
  }
  return HB_OK;
}

int cg_mixed(Context *c, int op, double kappa, double rho, double2 *x, const double2 *b, float rest,
             int maxiter, int log, int prec, double delta, int max_inner, int *iters, int *n_rel,
             double *true_rtr) {
  HB_CHECK(op == HB_OP_MTDAGMT || op == HB_OP_WDAGW, HB_E_ARG,
           "cg_mixed: operator must be HB_OP_MTDAGMT or HB_OP_WDAGW (got %d)", op);
  HB_CHECK(delta > 0.0 && delta < 1.0, HB_E_ARG, "cg_mixed: delta must be in (0, 1)");
  HB_CHECK(max_inner >= 1, HB_E_ARG, "cg_mixed: max_inner must be >= 1");
  HB_CHECK(maxiter >= 1, HB_E_ARG, "cg_mixed: maxiter must be >= 1");
  if (prec == HB_PREC_F64)
    return cg_f64(c, op, kappa, rho, x, b, rest, maxiter, log, iters, true_rtr);
  if (prec == HB_PREC_F32)
    return cg_mixed_impl<SF32, SF32>(c, op, kappa, rho, x, b, rest, maxiter, log, delta, max_inner, iters, n_rel, true_rtr);
  if (prec == HB_PREC_F16)
    return cg_mixed_impl<SF16, SF16>(c, op, kappa, rho, x, b, rest, maxiter, log, delta, max_inner, iters, n_rel, true_rtr);
  if (prec == HB_PREC_F16_GAUGE)
    return cg_mixed_impl<SF32, SF16>(c, op, kappa, rho, x, b, rest, maxiter, log, delta, max_inner, iters, n_rel, true_rtr);
  set_error("cg_mixed: precision %d (use 64, 32, 16 or 18)", prec);
  return HB_E_ARG;
}

// average time of the first half of the reduced-precision operator, the
// hopping kernel with the A_oo^-1 epilogue (out = A^-1 D in, odd output), on the
// context stream
template <class S>
int time_dslash_lp(Context *c, int reps, const double2 *in64, double *ms_out) {
  int rc = 0;
  SpinorPtr<S> in = SpinorAlloc<S>::get(c, SLOT_LP0, SLOT_LPN, &rc); HB_TRY(rc);
  SpinorPtr<S> out = SpinorAlloc<S>::get(c, SLOT_LP3, SLOT_LPN3, &rc); HB_TRY(rc);
  k_cvt_spinor<S><<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(in, in64, c->g.vh);
  HB_HIP(hipGetLastError());
  const bool clov = use_clover(c);
  DslashArgs<S, S> a{};
  a.g = c->g;
  a.out_parity = 1;
  a.out = out;
  a.in = in;
  a.U = LP<S>::gauge(c);
  a.C = clov ? LP<S>::clov(c, HB_CLOVER_AINV) : nullptr;
  a.Cn = clov ? LP<S>::norm(c, HB_CLOVER_AINV) : nullptr;
  for (int k = 0; k < 2; k++) HB_TRY(launch_dslash(a, false, EPI_CLINV, c->stream));
  EventTimer tm;
  HB_TRY(tm.create());
  HB_TRY(tm.start(c->stream));
  for (int k = 0; k < reps; k++) HB_TRY(launch_dslash(a, false, EPI_CLINV, c->stream));
  HB_TRY(tm.stop(c->stream));
  float ms = 0.f;
  HB_TRY(tm.elapsed(&ms));
  *ms_out = ms / reps;
  return HB_OK;
}

// the mixed solver's operator at reduced precision on an FP64 device spinor:
// in is stored at precision S (links and clover at G), the operator kernels of
// the inner iteration are applied (M~ or M~^+, with rho for W; M~^+ M~ or W^+ W
// as the solver chains them), and the stored result is decoded to FP64
template <class S, class G>
int apply_lp(Context *c, int op, double kappa, double rho, double2 *out64, const double2 *in64) {
  int rc = 0;
  SpinorPtr<S> in = SpinorAlloc<S>::get(c, SLOT_LP0, SLOT_LPN, &rc); HB_TRY(rc);
  SpinorPtr<S> out = SpinorAlloc<S>::get(c, SLOT_LP2, SLOT_LPN2, &rc); HB_TRY(rc);
  SpinorPtr<S> t = SpinorAlloc<S>::get(c, SLOT_LP3, SLOT_LPN3, &rc); HB_TRY(rc);
  SpinorPtr<S> y = SpinorAlloc<S>::get(c, SLOT_LP4, SLOT_LPN4, &rc); HB_TRY(rc);
  HB_TRY(ensure_lowprec(c, G::kBytes == 8 ? 32 : 16));
  const int vh = c->g.vh;
  k_cvt_spinor<S><<<nblocks(vh), kBlock, 0, c->stream>>>(in, in64, vh);
  HB_HIP(hipGetLastError());
  const bool w = op == HB_OP_W || op == HB_OP_W_DAG || op == HB_OP_WDAGW;
  const double r = w ? rho : 0.0;
  if (op == HB_OP_MTDAGMT || op == HB_OP_WDAGW) {
    HB_TRY((mtil_lp<S, G>(c, false, kappa, r, y, in, t, nullptr, SpinorPtr<S>{}, nullptr)));
    HB_TRY((mtil_lp<S, G>(c, true, kappa, r, out, y, t, nullptr, SpinorPtr<S>{}, nullptr)));
  } else {
    const bool dag = op == HB_OP_MTIL_DAG || op == HB_OP_W_DAG;
    HB_TRY((mtil_lp<S, G>(c, dag, kappa, r, out, in, t, nullptr, SpinorPtr<S>{}, nullptr)));
  }
  k_spinor_to_f64<S><<<nblocks(vh), kBlock, 0, c->stream>>>(out64, out, vh);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

}  // namespace hb

using namespace hb;

extern "C" {

int hb_time_dslash_lp(hb_context *ctx, int precision, int reps, const double *in_d, double *ms) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(in_d && ms, HB_E_ARG, "hb_time_dslash_lp: null pointer");
  HB_CHECK(reps >= 1, HB_E_ARG, "hb_time_dslash_lp: reps must be >= 1");
  HB_CHECK(precision == HB_PREC_F32 || precision == HB_PREC_F16, HB_E_ARG,
           "hb_time_dslash_lp: precision %d (use 32 or 16)", precision);
  HB_HIP(hipSetDevice(c->device));
  HB_TRY(ensure_lowprec(c, precision));
  const double2 *in = reinterpret_cast<const double2 *>(in_d);
  return precision == HB_PREC_F16 ? time_dslash_lp<SF16>(c, reps, in, ms)
                                  : time_dslash_lp<SF32>(c, reps, in, ms);
}

int hb_apply_lp_d(hb_context *ctx, int op, double kappa, double rho, int precision, double *out_d,
                  const double *in_d) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(out_d && in_d && out_d != in_d, HB_E_ARG, "hb_apply_lp_d: bad pointers");
  HB_CHECK(op >= HB_OP_MTIL && op <= HB_OP_WDAGW, HB_E_ARG, "hb_apply_lp_d: operator %d", op);
  HB_HIP(hipSetDevice(c->device));
  double2 *out = reinterpret_cast<double2 *>(out_d);
  const double2 *in = reinterpret_cast<const double2 *>(in_d);
  if (precision == HB_PREC_F32) return apply_lp<SF32, SF32>(c, op, kappa, rho, out, in);
  if (precision == HB_PREC_F16) return apply_lp<SF16, SF16>(c, op, kappa, rho, out, in);
  if (precision == HB_PREC_F16_GAUGE) return apply_lp<SF32, SF16>(c, op, kappa, rho, out, in);
  set_error("hb_apply_lp_d: precision %d (use 32, 16 or 18)", precision);
  return HB_E_ARG;
}

int hb_cg_mixed_d(hb_context *ctx, int op, double kappa, double rho, double *x_d, const double *b_d,
                  float rest, int maxiter, int log, int precision, double delta, int max_inner,
                  int *iters, int *n_reliable, double *true_rtr) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(x_d && b_d && x_d != b_d, HB_E_ARG, "hb_cg_mixed: bad pointers");
  HB_HIP(hipSetDevice(c->device));
  if (n_reliable) *n_reliable = 0;
  return cg_mixed(c, op, kappa, rho, reinterpret_cast<double2 *>(x_d), reinterpret_cast<const double2 *>(b_d),
                  rest, maxiter, log, precision, delta, max_inner, iters, n_reliable, true_rtr);
}

int hb_cg_mixed(hb_context *ctx, int op, double kappa, double rho, double *x, const double *b,
                float rest, int maxiter, int log, int precision, double delta, int max_inner,
                int *iters, int *n_reliable, double *true_rtr) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(x && b, HB_E_ARG, "hb_cg_mixed: null pointer");
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  double2 *dx = spinor_scratch(c, SLOT_X, &rc); HB_TRY(rc);
  double2 *db = spinor_scratch(c, SLOT_B, &rc); HB_TRY(rc);
  HB_TRY(spinor_upload(c, dx, x));
  HB_TRY(spinor_upload(c, db, b));
  if (n_reliable) *n_reliable = 0;
  int r = cg_mixed(c, op, kappa, rho, dx, db, rest, maxiter, log, precision, delta, max_inner,
                   iters, n_reliable, true_rtr);
  if (r != HB_OK && r != HB_E_NOCONV) return r;
  HB_TRY(spinor_download(c, x, dx));
  return r;
}

}  // extern "C"
