// hb_blas.h - spinor vector kernels, reductions and CG device state.
#pragma once

#include "hb_kernels.h"

namespace hb {

// Device-resident CG scalars (cg.F90:61-116); kernels read and update them so
// that an iteration needs no host round trip.  Every block of the p update
// forms the new scalars itself and one of them stores them, while the others
// may still be reading the old ones: iteration k reads slot k & 1 and writes
// the other.
struct CgSlot {
  double rtr;      // |r|^2 the iteration starts from (rtr_old)
  double last;     // |r|^2 it was left with (rtr)
  int iter;
  int done;        // 0 running, 1 converged, 2 maxiter reached
};
struct CgState {
  CgSlot s[2];
  double pap;      // <p, A p> of the iteration, from the r update for the p update
  double alpha[4]; // of the iterations whose x updates are pending (CgRing)
  double rest;     // stopping bound on |r|^2 (cg_para%rest, promoted to FP64)
  int maxiter;
  double res[4];   // scratch results (true residual etc.)
};

// finalize functor of the start (cg.F90:84-89): rtr_old = |r|^2
struct FinCgStart {
  CgState *st;
  __device__ void operator()(const double (&t)[1]) const {
    st->s[0] = CgSlot{t[0], t[0], 0, 0};
  }
};
struct FinStore1 {
  double *out;
  __device__ void operator()(const double (&t)[1]) const { out[0] = t[0]; }
};
struct FinStore2 {
  double *out;
  __device__ void operator()(const double (&t)[2]) const { out[0] = t[0]; out[1] = t[1]; }
};

int clover_mult_f64(Context *c, int which, int eo, double2 *out, const double2 *in);
// blocks of the linear CG vector kernels, and of their partial sums
inline int vector_grid(int vh) {
  const int n = nblocks(12 * vh);
  return n < 2048 ? n : 2048;
}
// `red`: per-block partial sums of the reductions (at least nblocks(vh)
// doubles); null selects the context's own buffer
int cg_init(Context *c, CgState *st, double rest, int maxiter);
int cg_start(Context *c, double2 *r, double2 *p, const double2 *b, CgState *st, double *red = nullptr);
// more than `most` partials (skip: as the kernel that left them) become one,
// at p + n; otherwise nothing happens
int shorten_partials(Context *c, const double *&p, int &n, const int *skip, int most = kMaxParts);
// the vector updates of iteration k: from the partials of <p, A p>
// (pa, na of them) to those of |r|^2 (pb, vector_grid(vh) doubles), and on
int cg_update(Context *c, double2 *r, const double2 *q, CgState *st, int k, const double *pa, int na, double *pb);
// Search directions: p of iteration k is p[k & 3].  Four buffers on lattices
// that are bound by the bytes of the updates: x then takes up four directions
// at a time, in the order and with the sums of one at a time (us per iteration
// with one / four: 141 k sites per parity 256.5 / 253.9, 160 k 279.5 / 276.9, 332 k
// 586.6 / 576.9).  One (all four the same) elsewhere, and where there is no memory for the others (spare()).
struct CgRing {
  double2 *p[4];
};
int cg_pupdate(Context *c, double2 *x, const CgRing &ring, const double2 *r, CgState *st, int k, const double *pb);
int residual(Context *c, double2 *out, const double2 *b, double *res_d, double *red = nullptr);
int dot_norm(Context *c, const double2 *x, const double2 *y, double *res_d);
int zero_f64(Context *c, double2 *p, size_t n);
int copy_f64(Context *c, double2 *d, const double2 *s, size_t n);

// host helpers from hb_fields.hip
int spinor_upload(Context *c, double2 *dst_d, const double *host);
int spinor_download(Context *c, double *host, const double2 *src_d);
int gen_upload(Context *c, double *dst_d, const double *host, int stride);
int gen_download(Context *c, double *host, const double *src_d, int stride);
int alloc_fp64_fields(Context *c);

}  // namespace hb
