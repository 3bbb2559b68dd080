// hb_blas.hip - spinor BLAS-1 with deterministic grid reductions, standalone
// clover multiplies, and precision conversions of spinors, links and clover.
#include "hb_blas.h"

#include "hb_dslash.h"

namespace hb {

// ---------------------------------------------------------------------------
// standalone clover multiplies (clover/clover_mult_a.F90, _ao, _b)
// ---------------------------------------------------------------------------
template <class S, int MODE>
__global__ __launch_bounds__(kBlock) void k_clover_mult(SpinorPtr<S> out, SpinorPtr<S> in,
                                                        const typename S::ST *C, const float *Cn,
                                                        int eo, int vh) {
  using V = typename S::V;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  V x[12], y[12];
  load_spinor<S>(x, in, i, vh);
  clover_apply<S, MODE>(y, x, C, Cn, eo, i, vh);
  store_spinor<S>(out, i, vh, y);
}

// out = A in (mode 0) or the LDL^+ solve (mode 1) with parity 0 of the FP64
// clover field C ([2][36][vh] device layout)
int clover_mult_parity_f64(Context *c, int mode, const double2 *C, double2 *out, const double2 *in) {
  SpinorPtr<SF64> o{out, nullptr}, s{const_cast<double2 *>(in), nullptr};
  if (mode == 1)
    k_clover_mult<SF64, 1><<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(o, s, C, nullptr, 0, c->g.vh);
  else
    k_clover_mult<SF64, 0><<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(o, s, C, nullptr, 0, c->g.vh);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int clover_mult_f64(Context *c, int which, int eo, double2 *out, const double2 *in) {
  SpinorPtr<SF64> o{out, nullptr}, s{const_cast<double2 *>(in), nullptr};
  if (which == HB_CLOVER_B)
    k_clover_mult<SF64, 1><<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(o, s, c->clov[which], nullptr, eo, c->g.vh);
  else
    k_clover_mult<SF64, 0><<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(o, s, c->clov[which], nullptr, eo, c->g.vh);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

// ---------------------------------------------------------------------------
// FP64 CG vector kernels (cg.F90:81-116); scalars live in CgState on device
// ---------------------------------------------------------------------------
// Vector kernels: one thread per site, the 12 components of a site in 12
// coalesced planes (component k of site i at k*vh + i).
#define HB_SITE_LOOP for (int k = 0; k < 12; k++)
#define HB_AT(ptr, k) (ptr)[(size_t)(k) * vh + i]
// r = b - r, p = r, rtr_old = |r|^2  (cg.F90:84-89)
__global__ __launch_bounds__(kBlock) void k_cg_start(double2 *__restrict__ r, double2 *__restrict__ p,
                                                     const double2 *__restrict__ b, int vh,
                                                     double *partials) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0.0;
  if (i < vh) {
#pragma unroll
    HB_SITE_LOOP {
      double2 bb = HB_AT(b, k), rr = HB_AT(r, k);
      double2 v = make_double2(bb.x - rr.x, bb.y - rr.y);
      HB_AT(r, k) = v;
      HB_AT(p, k) = v;
      s += v.x * v.x + v.y * v.y;
    }
  }
  double vals[1] = {s};
  block_partials<1>(vals, partials);
}

// The updates of an iteration have one thread per complex number, not per
// site: small lattices have too few sites to fill the chip.  NT: the results
// are streamed past the caches, as the hopping kernels' (store_spinor).
template <bool NT> __device__ __forceinline__ void st_cg(double2 *p, int i, double2 v) {
  if constexpr (NT) SF64::st_nt(p, i, v);
  else p[i] = v;
}
// alpha = rtr_old / pAp; r -= alpha q; rtr = |r|^2 (cg.F90:96-109).  The
// x update of the same iteration is done by k_cg_pupdate, which reads p anyway.
template <bool NT>
__global__ __launch_bounds__(kBlock) void k_cg_update(double2 *__restrict__ r, const double2 *__restrict__ q, int n,
                                                      CgState *st, int k, const double *pa, int na, double *pb) {
  const CgSlot c = st->s[k & 1];
  if (c.done) return;
  // the first operands are on their way while the partials are summed
  const int step = gridDim.x * blockDim.x;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double2 qq = i < n ? q[i] : double2{}, rr = i < n ? r[i] : double2{};
  asm volatile("" ::: "memory");
  const double pap = partials_total(pa, na);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->pap = pap;
  const double alpha = c.rtr / pap;
  double s = 0.0;
  while (i < n) {
    const double2 v = make_double2(rr.x - alpha * qq.x, rr.y - alpha * qq.y);
    s += v.x * v.x + v.y * v.y;
    const int j = i + step;
    if (j < n) {
      qq = q[j];
      rr = r[j];
    }
    st_cg<NT>(r, i, v);
    i = j;
  }
  double vals[1] = {s};
  block_partials<1>(vals, pb);
}

// x += alpha p of the iteration just finished (cg.F90:97-98), the stop test
// (cg.F90:111) and, unless the solve has ended, p = r + beta p (sc_xpby,
// sc.F90:184-201)
template <bool NT>
__global__ __launch_bounds__(kBlock) void k_cg_pupdate(double2 *__restrict__ x, double2 *__restrict__ p,
                                                       const double2 *__restrict__ r, int n, CgState *st, int k,
                                                       const double *pb, int nb, Note note) {
  const CgSlot c = st->s[k & 1];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (c.done) {
    if (first) {
      st->s[~k & 1] = c;
      note.tell(c.done);
    }
    return;
  }
  const int step = gridDim.x * blockDim.x;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double2 pp = i < n ? p[i] : double2{}, xx = i < n ? x[i] : double2{}, rr = i < n ? r[i] : double2{};
  asm volatile("" ::: "memory");
  const double rtr = partials_total(pb, nb);
  const double alpha = c.rtr / st->pap, beta = rtr / c.rtr;
  const int iter = c.iter + 1;
  const int done = rtr <= st->rest ? 1 : iter >= st->maxiter ? 2 : 0;
  if (first) {
    st->s[~k & 1] = CgSlot{done ? c.rtr : rtr, rtr, iter, done};
    note.tell(done);
  }
  while (i < n) {
    const double2 xv = make_double2(xx.x + alpha * pp.x, xx.y + alpha * pp.y);
    const double2 pv = make_double2(rr.x + beta * pp.x, rr.y + beta * pp.y);
    const int j = i + step;
    if (j < n) {
      pp = p[j];
      xx = x[j];
      rr = r[j];
    }
    st_cg<NT>(x, i, xv);
    if (!done) st_cg<NT>(p, i, pv);
    i = j;
  }
}

// the same with the search directions in a ring (CgRing): 24^3x48 44.7 us
// against 49.3
__global__ __launch_bounds__(kBlock) void k_cg_pupdate_ring(double2 *__restrict__ x, CgRing ring,
                                                            const double2 *__restrict__ r, int n, CgState *st, int k,
                                                            const double *pb, int nb, Note note) {
  const CgSlot c = st->s[k & 1];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (c.done) {
    if (first) {
      st->s[~k & 1] = c;
      note.tell(c.done);
    }
    return;
  }
  const int slot = k & 3;
  const double *alphas = st->alpha;
  const double rtr = partials_total(pb, nb);
  const double alpha = c.rtr / st->pap, beta = rtr / c.rtr;
  const int iter = c.iter + 1;
  const int done = rtr <= st->rest ? 1 : iter >= st->maxiter ? 2 : 0;
  if (first) {
    st->s[~k & 1] = CgSlot{done ? c.rtr : rtr, rtr, iter, done};
    st->alpha[slot] = alpha;
    note.tell(done);
  }
  const bool take = slot == 3 || done;
  const double2 *p = ring.p[slot];
  double2 *pn = ring.p[(k + 1) & 3];
  double al[3];
  for (int q = 0; q < 3; q++) al[q] = q < slot ? alphas[q] : 0.0;
#pragma unroll 2
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double2 pp = p[i];
    if (take) {
      double2 xx = x[i];
      for (int q = 0; q < slot; q++) {
        const double2 v = ring.p[q][i];
        xx.x += al[q] * v.x; xx.y += al[q] * v.y;
      }
      xx.x += alpha * pp.x; xx.y += alpha * pp.y;
      SF64::st_nt(x, i, xx);
    }
    if (!done) {
      const double2 rr = r[i];
      SF64::st_nt(pn, i, make_double2(rr.x + beta * pp.x, rr.y + beta * pp.y));
    }
  }
}

// out = b - out, result |out|^2
__global__ __launch_bounds__(kBlock) void k_residual(double2 *__restrict__ out, const double2 *__restrict__ b,
                                                     int vh, double *partials) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0.0;
  if (i < vh) {
#pragma unroll
    HB_SITE_LOOP {
      double2 bb = HB_AT(b, k), o = HB_AT(out, k);
      double2 v = make_double2(bb.x - o.x, bb.y - o.y);
      HB_AT(out, k) = v;
      s += v.x * v.x + v.y * v.y;
    }
  }
  double vals[1] = {s};
  block_partials<1>(vals, partials);
}

// Re<x, y> and |x|^2 of FP64 fields
__global__ __launch_bounds__(kBlock) void k_dot_norm(const double2 *__restrict__ x, const double2 *__restrict__ y,
                                                     int vh, double *partials) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s0 = 0.0, s1 = 0.0;
  if (i < vh) {
#pragma unroll
    HB_SITE_LOOP {
      double2 a = HB_AT(x, k), b = HB_AT(y, k);
      s0 += a.x * b.x + a.y * b.y;
      s1 += a.x * a.x + a.y * a.y;
    }
  }
  double vals[2] = {s0, s1};
  block_partials<2>(vals, partials);
}

#undef HB_SITE_LOOP
#undef HB_AT

__global__ void k_zero(double2 *p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t k = i; k < n; k += (size_t)gridDim.x * blockDim.x) p[k] = make_double2(0.0, 0.0);
}

__global__ void k_copy(double2 *__restrict__ d, const double2 *__restrict__ s, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t k = i; k < n; k += (size_t)gridDim.x * blockDim.x) d[k] = s[k];
}

// every field of the CG state cleared, then the stopping bound and maxiter
__global__ void k_cg_init(CgState *st, double rest, int maxiter) {
  if (threadIdx.x == 0) {
    CgState s{};
    s.rest = rest;
    s.maxiter = maxiter;
    *st = s;
  }
}

int cg_init(Context *c, CgState *st, double rest, int maxiter) {
  k_cg_init<<<1, 64, 0, c->stream>>>(st, rest, maxiter);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int cg_start(Context *c, double2 *r, double2 *p, const double2 *b, CgState *st, double *red) {
  const int vh = c->g.vh, grid = nblocks(vh);
  if (!red) red = c->red;
  k_cg_start<<<grid, kBlock, 0, c->stream>>>(r, p, b, vh, red);
  k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(red, grid, nullptr, FinCgStart{st});
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int shorten_partials(Context *c, const double *&p, int &n, const int *skip, int most) {
  if (n <= most) return HB_OK;
  double *out = const_cast<double *>(p) + n;
  k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(p, n, skip, FinStore1{out});
  HB_HIP(hipGetLastError());
  p = out;
  n = 1;
  return HB_OK;
}

int cg_update(Context *c, double2 *r, const double2 *q, CgState *st, int k, const double *pa, int na, double *pb) {
  const int vh = c->g.vh;
  const auto f = operator_policy<SF64, SF64R>(vh) == kNT ? k_cg_update<true> : k_cg_update<false>;
  f<<<vector_grid(vh), kBlock, 0, c->stream>>>(r, q, 12 * vh, st, k, pa, na, pb);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int cg_pupdate(Context *c, double2 *x, const CgRing &ring, const double2 *r, CgState *st, int k, const double *pb) {
  const int vh = c->g.vh;
  if (ring.p[1] != ring.p[0]) {
    k_cg_pupdate_ring<<<vector_grid(vh), kBlock, 0, c->stream>>>(x, ring, r, 12 * vh, st, k, pb, vector_grid(vh),
                                                               next_note(c));
  } else {
    const auto f = operator_policy<SF64, SF64R>(vh) == kNT ? k_cg_pupdate<true> : k_cg_pupdate<false>;
    f<<<vector_grid(vh), kBlock, 0, c->stream>>>(x, ring.p[0], r, 12 * vh, st, k, pb, vector_grid(vh), next_note(c));
  }
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int residual(Context *c, double2 *out, const double2 *b, double *res_d, double *red) {
  const int vh = c->g.vh, grid = nblocks(vh);
  if (!red) red = c->red;
  k_residual<<<grid, kBlock, 0, c->stream>>>(out, b, vh, red);
  k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(red, grid, nullptr, FinStore1{res_d});
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int dot_norm(Context *c, const double2 *x, const double2 *y, double *res_d) {
  const int vh = c->g.vh, grid = nblocks(vh);
  k_dot_norm<<<grid, kBlock, 0, c->stream>>>(x, y, vh, c->red);
  k_finalize<2><<<1, kFinThreads, 0, c->stream>>>(c->red, grid, nullptr, FinStore2{res_d});
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int zero_f64(Context *c, double2 *p, size_t n) {
  k_zero<<<nblocks((int)std::min<size_t>(n, (size_t)1 << 24)), kBlock, 0, c->stream>>>(p, n);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int copy_f64(Context *c, double2 *d, const double2 *s, size_t n) {
  k_copy<<<nblocks((int)std::min<size_t>(n, (size_t)1 << 24)), kBlock, 0, c->stream>>>(d, s, n);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

}  // namespace hb
