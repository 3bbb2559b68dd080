// hb_force.hip - fermion force (dsf.F90 + d/DSFxyzt.F90 + clover/clover_d.F90),
// clover-determinant force (dsd.F90, clover_dsd), Wilson gauge force
// (dsg.F90), link update (hmc_u.F90) and the clover action
// (clover/clover_action.F90), all in FP64 on device-resident fields.
//
// The force kernels gather: all terms of a link are added to its 8 momentum
// coordinates by one thread, so no atomics are needed and the result is
// deterministic.  In the fermion and clover forces one thread owns one link
// (mu, eo, i); in the gauge force a wave owns a plane of 64 sites, and the
// shares of the six planes meet in LDS.  Momenta are device SoA
// P[4 mu][2 eo][8][vh].
#include "hb_ops.h"
#include "hb_su3.h"

namespace hb {

// ---------------------------------------------------------------------------
// spinor access helpers (FP64 SoA, component k = 3*spin + colour)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ld_spinor(double2 (&v)[12], const double2 *__restrict__ f, int i, int vh) {
#pragma unroll
  for (int k = 0; k < 12; k++) v[k] = f[(size_t)k * vh + i];
}

__device__ __forceinline__ double *mom(double *P, int mu, int eo, int vh) {
  return P + (size_t)((mu * 2 + eo) * 8) * vh;
}
__device__ __forceinline__ void mom_add(double *P, int mu, int eo, int i, int vh, const double (&q)[8]) {
  double *b = mom(P, mu, eo, vh) + i;
#pragma unroll
  for (int j = 0; j < 8; j++) b[(size_t)j * vh] += q[j];
}

// ---------------------------------------------------------------------------
// hopping part of the fermion force (dsf.F90:77-98 with DSFxyzt.F90:77-117)
// ---------------------------------------------------------------------------
// The half spinor of the projector (1 + SG gamma_MU), index 2*colour + spin.
// ((1 + SG gamma) a) (x) conj(b), summed over the four spins, is the sum over
// two of h(a) (x) conj(h(b)): gamma is Hermitian and the projector of rank two.
template <int MU, int SG>
__device__ __forceinline__ void half_spinor(double2 (&h)[6], const SpinorView<SF64> &f, int i) {
  if constexpr (MU == 3) {
    double2 p[6];
    f.load_pair_raw(p, i, SG < 0 ? 2 : 0);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      h[2 * c] = p[c];
      h[2 * c + 1] = p[3 + c];
    }
  } else {
    double2 p[12];
    f.load(p, i);
    project<MU, SG>(h, p);
  }
}

// q += s Im Tr(lambda_j x y^+), x and y 3 x 2
__device__ __forceinline__ void im_tr_j_outer(double (&q)[8], const double2 (&x)[6], const double2 (&y)[6], double s) {
  M3 v;
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      double2 t = make_double2(0.0, 0.0);
      cfma3<false, true>(t, x[2 * a], y[2 * b]);
      cfma3<false, true>(t, x[2 * a + 1], y[2 * b + 1]);
      v.m[3 * a + b] = t;
    }
  im_tr_j(q, v, s);
}

// Bvec/Avec of parity E (index 0) and of the other parity (index 1):
// E = EVEN: forward term (b_i, at_j), backward (a_i, bt_j);
// E = ODD : forward term (bt_i, a_j), backward (at_i, b_j).
// The link multiplies a half spinor, before the outer product with the other.
template <int MU>
__device__ void hop_force_link(double (&q)[8], const double2 *__restrict__ U, const Geom &g, int e, int i,
                               const int (&x)[4], const double2 *Bi, const double2 *Aj,
                               const double2 *Ai, const double2 *Bj, double s) {
  const int vh = g.vh;
  int c[4] = {x[0], x[1], x[2], x[3]};
  double sg = MU == 3 ? 2.0 * s : s;  // the t projector's factor 2
  c[MU] += 1;
  if (c[MU] == g.L[MU]) { c[MU] = 0; sg *= (double)g.bc[MU]; }  // flip_bc's sign of the link
  const int j = site_index(g, c[0], c[1], c[2], c[3]);
  const M3 u = link_b(U, MU, e, i, vh);
  const auto view = [vh](const double2 *f) {
    return SpinorView<SF64>(SpinorPtr<SF64>{const_cast<double2 *>(f), nullptr}, vh);
  };
  double2 h[6], k[6], w[6];
  // forward: p -= s Im Tr(lambda U w), w = ((1 - g) A_j) (x) conj(B_i)
  half_spinor<MU, -1>(h, view(Aj), j);
  half_spinor<MU, -1>(k, view(Bi), i);
  su3_mul_half(w, u.m, h);
  im_tr_j_outer(q, w, k, -sg);
  __builtin_amdgcn_sched_barrier(0);
  // backward: p += s Im Tr(lambda w U^+), w = ((1 + g) A_i) (x) conj(B_j)
  half_spinor<MU, 1>(h, view(Ai), i);
  half_spinor<MU, 1>(k, view(Bj), j);
  su3_mul_half(w, u.m, k);
  im_tr_j_outer(q, h, w, sg);
}

// spinors of the hopping force: a, b on the even sites, at = A~, bt = B~ on the
// odd ones; s = 0: no hopping force
struct HopForce {
  const double2 *a, *b, *at, *bt;
  double s;
};
__device__ __forceinline__ void hop_force(double (&q)[8], const double2 *__restrict__ U, const Geom &g, int mu, int e,
                                          int i, const int (&x)[4], const HopForce &h) {
  const double2 *Bi = e == 0 ? h.b : h.bt, *Aj = e == 0 ? h.at : h.a;
  const double2 *Ai = e == 0 ? h.a : h.at, *Bj = e == 0 ? h.bt : h.b;
  switch (mu) {
    case 0: hop_force_link<0>(q, U, g, e, i, x, Bi, Aj, Ai, Bj, h.s); break;
    case 1: hop_force_link<1>(q, U, g, e, i, x, Bi, Aj, Ai, Bj, h.s); break;
    case 2: hop_force_link<2>(q, U, g, e, i, x, Bi, Aj, Ai, Bj, h.s); break;
    default: hop_force_link<3>(q, U, g, e, i, x, Bi, Aj, Ai, Bj, h.s); break;
  }
}

// ---------------------------------------------------------------------------
// clover parts.  The six sigma_mu_nu fields w_k of clover_bsa / clover_ts
// (planes k = 12, 13, 14, 23, 24, 34) enter the derivative of the clover
// leaves (clover_d) once for each orientation of a leaf, as w and as w^+ on
// the reversed path, so only the Hermitian H_k = s (w_k + w_k^+) is needed;
// the scale s of the force is part of it.
// ---------------------------------------------------------------------------
// s (w + w^+) of a general w
__device__ __forceinline__ H3 herm(const M3 &w, double s) {
  H3 h;
  h.d[0] = 2.0 * s * w.m[0].x;
  h.d[1] = 2.0 * s * w.m[4].x;
  h.d[2] = 2.0 * s * w.m[8].x;
  h.o[0] = cscale<double2>(s, cadd(w.m[1], cconj(w.m[3])));
  h.o[1] = cscale<double2>(s, cadd(w.m[2], cconj(w.m[6])));
  h.o[2] = cscale<double2>(s, cadd(w.m[5], cconj(w.m[7])));
  return h;
}
// w_k = sum over spins of (S_k a)_s (x) conj(b_s) (clover_bsa_12..34) from the
// sixteen products T(s, s') = a_s' (x) conj(b_s): S_k has one entry per row,
//   12: -00 +11 -22 +33    13: i (10 - 01 + 32 - 23)   23: -(01 + 10 + 23 + 32)
//   14: 03 + 12 + 21 + 30  24: i (12 - 03 + 30 - 21)   34: 02 - 13 + 20 - 31
// (blockIdx.y: one of up to two fields)
struct HSpinors {
  double *F;
  const double2 *b, *a;
  double s;
};
__global__ __launch_bounds__(kBlock) void k_h_spinors(HSpinors h0, HSpinors h1, int vh) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  const HSpinors h = blockIdx.y == 0 ? h0 : h1;
  double *F = h.F;
  const double2 *b = h.b, *a = h.a;
  const double s = h.s;
  double2 av[12], bv[12];
  ld_spinor(av, a, i, vh);
  ld_spinor(bv, b, i, vh);
  // t += or -= a_s' (x) conj(b_s)
  const auto add = [&](M3 &t, int sb, int sa, double sign) {
#pragma unroll
    for (int ca = 0; ca < 3; ca++)
#pragma unroll
      for (int cb = 0; cb < 3; cb++) {
        const double2 z = make_double2(sign * av[3 * sa + ca].x, sign * av[3 * sa + ca].y);
        cfma3<false, true>(t.m[3 * ca + cb], z, bv[3 * sb + cb]);
      }
  };
  // both combinations of a pair of planes: f - e times i, and +-(e + f)
  const auto pair = [&](const M3 &e, const M3 &f, int ki, int kr, double sr) {
    M3 w;
#pragma unroll
    for (int m = 0; m < 9; m++) w.m[m] = ci(csub(f.m[m], e.m[m]));
    store_h(F, ki, i, vh, herm(w, s));
#pragma unroll
    for (int m = 0; m < 9; m++) w.m[m] = cadd(e.m[m], f.m[m]);
    store_h(F, kr, i, vh, herm(w, sr * s));
  };
  {
    M3 w = m3_zero();
    add(w, 0, 0, -1.0); add(w, 1, 1, 1.0); add(w, 2, 2, -1.0); add(w, 3, 3, 1.0);
    store_h(F, 0, i, vh, herm(w, s));
  }
  {
    M3 e = m3_zero(), f = m3_zero();
    add(e, 0, 1, 1.0); add(e, 2, 3, 1.0);
    add(f, 1, 0, 1.0); add(f, 3, 2, 1.0);
    pair(e, f, 1, 3, -1.0);
  }
  {
    M3 e = m3_zero(), f = m3_zero();
    add(e, 0, 3, 1.0); add(e, 2, 1, 1.0);
    add(f, 1, 2, 1.0); add(f, 3, 0, 1.0);
    pair(e, f, 4, 2, 1.0);
  }
  {
    M3 w = m3_zero();
    add(w, 0, 2, 1.0); add(w, 1, 3, -1.0); add(w, 2, 0, 1.0); add(w, 3, 1, -1.0);
    store_h(F, 5, i, vh, herm(w, s));
  }
}

// Z = (L D L^+)^-1 of one stored block (L unit lower triangular, D_k the
// stored 1/2 * 1/d_k), upper triangle: M = L^-1, Z_rc = sum_k conj(M_kr) D_k M_kc
__device__ __forceinline__ void ldl6_inverse(double2 (&Z)[6][6], const double2 (&w)[18]) {
  double2 M[6][6];
  const double d[6] = {w[15].x, w[15].y, w[16].x, w[16].y, w[17].x, w[17].y};
#pragma unroll
  for (int c = 0; c < 6; c++)
#pragma unroll
    for (int r = c + 1; r < 6; r++) {
      double2 t = w[r * (r - 1) / 2 + c];
#pragma unroll
      for (int k = c + 1; k < r; k++) cfma3<false, false>(t, w[r * (r - 1) / 2 + k], M[k][c]);
      M[r][c] = make_double2(-t.x, -t.y);
    }
#pragma unroll
  for (int r = 0; r < 6; r++)
#pragma unroll
    for (int c = r; c < 6; c++) {
      // k = c first: M_cc = 1
      double2 t = r == c ? make_double2(d[c], 0.0) : cscale<double2>(d[c], cconj(M[c][r]));
#pragma unroll
      for (int k = c + 1; k < 6; k++) cfma3<true, false>(t, cscale<double2>(d[k], M[k][r]), M[k][c]);
      Z[r][c] = t;
    }
}

// H_k of T = A^-1 (clover_t_init, clover_ts) from the LDL^+ field of parity eo.
// T's spin blocks are T_uu = T_ll = Z_1 + Z_2 and T_ul = T_lu = Z_1 - Z_2 with
// the inverses Z of the two chiral blocks, so that with P = Z_1 + Z_2 and
// Q = Z_1 - Z_2 (2 x 2 spin blocks of 3 x 3 matrices)
//   w_12 = 2 (P_11 - P_00)  w_13 = 2i (P_01 - P_10)  w_23 = -2 (P_01 + P_10)
//   w_14 = 2 (Q_01 + Q_10)  w_24 = 2i (Q_01 - Q_10)  w_34 = 2 (Q_00 - Q_11)
__global__ __launch_bounds__(kBlock) void k_h_inverse(double *__restrict__ F, const double2 *__restrict__ Cb, int eo,
                                                      int vh, double s) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  double2 P[6][6], Q[6][6];
  {
    double2 w[18];
    load_clover_block<SF64>(w, Cb, nullptr, eo, 0, i, vh);
    ldl6_inverse(P, w);
  }
  {
    double2 w[18], z[6][6];
    load_clover_block<SF64>(w, Cb, nullptr, eo, 1, i, vh);
    ldl6_inverse(z, w);
#pragma unroll
    for (int r = 0; r < 6; r++)
#pragma unroll
      for (int c = r; c < 6; c++) {
        Q[r][c] = csub(P[r][c], z[r][c]);
        P[r][c] = cadd(P[r][c], z[r][c]);
      }
  }
  // 4 s (X_11 - X_00) or its negative, X Hermitian: from the upper triangle
  const auto diag = [&](const double2 (&X)[6][6], int k, double f) {
    H3 h;
#pragma unroll
    for (int c = 0; c < 3; c++) h.d[c] = f * (X[3 + c][3 + c].x - X[c][c].x);
    h.o[0] = cscale<double2>(f, csub(X[3][4], X[0][1]));
    h.o[1] = cscale<double2>(f, csub(X[3][5], X[0][2]));
    h.o[2] = cscale<double2>(f, csub(X[4][5], X[1][2]));
    store_h(F, k, i, vh, h);
  };
  // X_01 =: Y: 4i s (Y - Y^+) and 4 fr s (Y + Y^+)
  const auto off = [&](const double2 (&X)[6][6], int ki, int kr, double fr) {
    M3 y, w;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) y.m[3 * a + b] = X[a][3 + b];
#pragma unroll
    for (int m = 0; m < 9; m++) w.m[m] = ci(y.m[m]);
    store_h(F, ki, i, vh, herm(w, 4.0 * s));  // i (Y - Y^+) = iY + (iY)^+
    store_h(F, kr, i, vh, herm(y, 4.0 * fr * s));
  };
  diag(P, 0, 4.0 * s);
  off(P, 1, 3, -1.0);
  off(Q, 4, 2, 1.0);
  diag(Q, 5, -4.0 * s);
}

// r += H a (LEFT) or a H
template <bool LEFT>
__device__ __forceinline__ void h_prod_acc(M3 &r, const H3 &h, const M3 &a) {
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) {
      double2 &t = r.m[3 * i + j];
      const double d = LEFT ? h.d[i] : h.d[j];
      t.x = fma(d, a.m[3 * i + j].x, t.x);
      t.y = fma(d, a.m[3 * i + j].y, t.y);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const int p = LEFT ? i : k, q = LEFT ? k : j;  // H_pq
        if (p == q) continue;
        const double2 x = LEFT ? a.m[3 * k + j] : a.m[3 * i + k];
        if (p < q) cfma3<false, false>(t, h.o[p + q - 1], x);
        else cfma3<true, false>(t, h.o[p + q - 1], x);
      }
    }
}
// The four products of a leaf pair below.  The inner product is formed a row
// or column at a time, so that no third matrix of temporaries is live.
//   S += l (c b)^+
__device__ __forceinline__ void acc_l_cb(M3 &S, const M3 &l, const M3 &c, const M3 &b) {
#pragma unroll
  for (int j = 0; j < 3; j++) {
    double2 t[3];
#pragma unroll
    for (int k = 0; k < 3; k++) t[k] = m3_elem<0>(c, b, j, k);
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int k = 0; k < 3; k++) cfma3<false, true>(S.m[3 * i + j], l.m[3 * i + k], t[k]);
    pin(S);
  }
}
//   S += (a b^+) l^+
__device__ __forceinline__ void acc_ab_l(M3 &S, const M3 &a, const M3 &b, const M3 &l) {
#pragma unroll
  for (int i = 0; i < 3; i++) {
    double2 t[3];
#pragma unroll
    for (int k = 0; k < 3; k++) t[k] = m3_elem<2>(a, b, i, k);
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int k = 0; k < 3; k++) cfma3<false, true>(S.m[3 * i + j], t[k], l.m[3 * j + k]);
    pin(S);
  }
}
//   S += l^+ (b^+ c)
__device__ __forceinline__ void acc_ld_bdc(M3 &S, const M3 &l, const M3 &b, const M3 &c) {
#pragma unroll
  for (int j = 0; j < 3; j++) {
    double2 t[3];
#pragma unroll
    for (int k = 0; k < 3; k++) t[k] = m3_elem<1>(b, c, k, j);
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int k = 0; k < 3; k++) cfma3<true, false>(S.m[3 * i + j], l.m[3 * k + i], t[k]);
    pin(S);
  }
}
//   S += (b a)^+ l
__device__ __forceinline__ void acc_bad_l(M3 &S, const M3 &b, const M3 &a, const M3 &l) {
#pragma unroll
  for (int i = 0; i < 3; i++) {
    double2 t[3];
#pragma unroll
    for (int k = 0; k < 3; k++) t[k] = m3_elem<0>(b, a, k, i);
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int k = 0; k < 3; k++) cfma3<true, false>(S.m[3 * i + j], t[k], l.m[3 * k + j]);
    pin(S);
  }
}

// the H pair of a dressed link: H(y) and H(y + nu), where their parity has a
// field, times sg = +-1
template <bool Y, bool N>
struct HPair {
  H3 y, n;
  __device__ __forceinline__ HPair(const double *Hy, int iy, const double *Hn, int in, int k, int vh) {
    if constexpr (Y) y = load_h(Hy, k, iy, vh);
    if constexpr (N) n = load_h(Hn, k, in, vh);
  }
  __device__ __forceinline__ static H3 times(const H3 &h, double s) {
    H3 r;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      r.o[q] = cscale<double2>(s, h.o[q]);
      r.d[q] = h.d[q] * s;
    }
    return r;
  }
  // L(y) = H(y) a + a H(y + nu) of the link a = U_nu(y)
  __device__ __forceinline__ M3 dress(const M3 &a, double sg) const {
    M3 r = m3_zero();
    if constexpr (Y) h_prod_acc<true>(r, times(y, sg), a);
    if constexpr (N) h_prod_acc<false>(r, times(n, sg), a);
    return r;
  }
};

// All clover_d contributions (clover/clover_d.F90:152-266) of one link: H0 and
// H1 are the H fields of the even and the odd sites (null: none).
//
// For the link U = U_mu(x) and a plane partner nu the leaf above is U A B C
// with A = U_nu(x+mu), B = U_mu(x+nu)^+, C = U_nu(x)^+, and the derivative
// takes H at its four corners; with L_nu(y) = H(y) U_nu(y) + U_nu(y) H(y+nu)
// their sum is
//   S_above = L_nu(x+mu) (U_nu(x) U_mu(x+nu))^+ + U_nu(x+mu) U_mu(x+nu)^+ L_nu(x)^+
//   S_below = L_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)
//             + (U_mu(x-nu) U_nu(x+mu-nu))^+ L_nu(x-nu)
// and the force is Re Tr(lambda U sum_nu +-(S_above - S_below)): 16 matrix
// products per plane for both parities together and one trace per link, where
// the leaves of each parity and orientation taken apart need 37 and 16.
//
// FP64 issue alone is 78 us of the fermion force's 138 us at 16^3x32 (both
// parities; 693 us leaf by leaf).  The rest is the latency of the loads, at
// two waves per SIMD: the operands of a step are therefore fetched during the
// step before, in 250 registers (fetched when needed, in 178 registers and
// still two waves, it took 193 us; one wave with 360 registers 181 us).  The
// parities that carry a field are template arguments: tested inside the steps,
// they split them into blocks across which the compiler keeps 100 registers more.
template <bool E, bool O>  // H on the link's parity, on the other
__device__ __forceinline__ void clover_leaves(M3 &S, const double2 *__restrict__ U, const Geom &g, int mu, int e, int i,
                                              const int (&x)[4], const double *He, const double *Ho) {
  const int o = 1 - e, vh = g.vh;
  const int id = nb(g, x[0], x[1], x[2], x[3], mu, 1);
#pragma unroll 1
  for (int nu = 0; nu < 4; nu++) {
    if (nu == mu) continue;
    const int lo = mu < nu ? mu : nu, hi = mu < nu ? nu : mu;
    const int k = lo == 0 ? hi - 1 : lo + hi;  // plane (lo, hi): 01 02 03 12 13 23
    const double sg = mu < nu ? 1.0 : -1.0;
    const int in = nb(g, x[0], x[1], x[2], x[3], nu, 1);
    const int idn = nb2(g, x[0], x[1], x[2], x[3], mu, 1, nu, 1);
    const int im = nb(g, x[0], x[1], x[2], x[3], nu, -1);
    const int idm = nb2(g, x[0], x[1], x[2], x[3], mu, 1, nu, -1);
    // every step's operands are loaded while the step before it computes
    const M3 a = link_b(U, nu, o, id, vh);
    const HPair<O, E> ha(Ho, id, He, idn, k, vh);
    const M3 b = link_b(U, mu, o, in, vh), c = link_b(U, nu, e, i, vh);
    M3 l = ha.dress(a, sg);
    step_end(l);
    const HPair<E, O> hc(He, i, Ho, in, k, vh);
    acc_l_cb(S, l, c, b);
    step_end(S);
    l = hc.dress(c, sg);
    step_end(l);
    const M3 a2 = link_b(U, nu, e, idm, vh);
    const HPair<E, O> ha2(He, idm, Ho, fresh(id), k, vh);
    acc_ab_l(S, a, b, l);
    step_end(S);
    const M3 b2 = link_b(U, mu, o, im, vh), c2 = link_b(U, nu, o, im, vh);
    l = ha2.dress(a2, -sg);
    step_end(l);
    const HPair<O, E> hc2(Ho, im, He, fresh(i), k, vh);
    acc_ld_bdc(S, l, b2, c2);
    step_end(S);
    l = hc2.dress(c2, -sg);
    step_end(l);
    acc_bad_l(S, b2, a2, l);
    step_end(S);
  }
}

// the clover force of one link and, for the fermion force, its hopping force
// (HOP; the spinors of hop): in a kernel of its own the hopping force reads the
// links and updates the momenta once more
template <bool HOP>
__global__ __launch_bounds__(kLinkBlock, 2) void k_clover_force(double *P, const double2 *__restrict__ U, Geom g, int run,
                                                                const double *H0, const double *H1, HopForce hop) {
  int mu, e, i;
  if (!link_slot(g, run, mu, e, i)) return;
  const double *He = e == 0 ? H0 : H1, *Ho = e == 0 ? H1 : H0;
  int x[4];
  site_coords(g, e, i, x[0], x[1], x[2], x[3]);
  double q[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (He || Ho) {
    M3 S = m3_zero();
    if (He && Ho) clover_leaves<true, true>(S, U, g, mu, e, i, x, He, Ho);
    else if (He) clover_leaves<true, false>(S, U, g, mu, e, i, x, He, Ho);
    else clover_leaves<false, true>(S, U, g, mu, e, i, x, He, Ho);
    re_tr_j_prod<0>(q, link_b(U, mu, e, i, g.vh), S, 1.0);
  }
  if (HOP && hop.s != 0.0) hop_force(q, U, g, mu, e, i, x, hop);
  mom_add(P, mu, e, i, g.vh, q);
}

// ---------------------------------------------------------------------------
// gauge force (dsg.F90:28-63) with the staple of staple.F90:28-76
// ---------------------------------------------------------------------------
// One wave per plane (mu, nu) of 64 sites.  The plaquette at x is the staple
// above for both of its links (v for U_mu(x), v^+ for U_nu(x)), which leaves
// ten links and nine products per plane, where the two links' staples taken
// apart read fourteen; the sites' own links, which every plane needs, are
// shared through LDS, and so are the six waves' shares of the four forces.
// No unit is saturated (vector memory addresser 59 % busy, 77 % with the own
// links in memory; FP64 issue 37 %): 32^3x64 1.30 ms, one wave per direction
// 1.54 ms; 16^3x32 118 -> 87 us.  Registers for one link fetched ahead spill
// (1.37 ms); two waves per SIMD with both own links held: 1.67 ms.
constexpr int kPlaneBlock = 384;
__global__ __launch_bounds__(kPlaneBlock, 3) void k_gauge_force(double *P, const double2 *__restrict__ U, Geom g, int run,
                                                                double s) {
  __shared__ union {
    double2 own[4][9][64];
    double part[6][2][8][64];
  } lds;
  int k, e, i;
  const bool active = link_slot(g, run, k, e, i);
  const int mu = k < 3 ? 0 : k < 5 ? 1 : 2, nu = k < 3 ? k + 1 : k < 5 ? k - 1 : 3;
  const int vh = g.vh, o = 1 - e, lane = threadIdx.x & 63;
  int x[4] = {0, 0, 0, 0};
  M3 t = m3_zero();
  if (active) {
    if (k < 4) {
      const M3 u = link_b(U, k, e, i, vh);
#pragma unroll
      for (int m = 0; m < 9; m++) lds.own[k][m][lane] = u.m[m];
    }
    site_coords(g, e, i, x[0], x[1], x[2], x[3]);
    const int xp = nb(g, x[0], x[1], x[2], x[3], mu, 1), yp = nb(g, x[0], x[1], x[2], x[3], nu, 1);
    t = m3_muld(link_b(U, nu, o, xp, vh), link_b(U, mu, o, yp, vh));
  }
  __syncthreads();
  double q[8] = {0, 0, 0, 0, 0, 0, 0, 0}, r[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (active) {
    const auto own = [&](int d) {
      M3 u;
#pragma unroll
      for (int m = 0; m < 9; m++) u.m[m] = lds.own[d][m][lane];
      return u;
    };
    const int xm = nb(g, x[0], x[1], x[2], x[3], mu, -1), ym = nb(g, x[0], x[1], x[2], x[3], nu, -1);
    const int xpym = nb2(g, x[0], x[1], x[2], x[3], mu, 1, nu, -1);
    const int xmyp = nb2(g, x[0], x[1], x[2], x[3], mu, -1, nu, 1);
    t = m3_muld(t, own(nu));
    step_end(t);
    im_tr_j(q, m3_mul(own(mu), t), s);
#pragma unroll
    for (int j = 0; j < 8; j++) r[j] = -q[j];
    t = m3_mul(link_b(U, mu, o, ym, vh), link_b(U, nu, e, xpym, vh));
    step_end(t);
    t = m3_dmul(t, link_b(U, nu, o, ym, vh));
    step_end(t);
    im_tr_j(q, m3_mul(own(mu), t), s);
    t = m3_mul(link_b(U, nu, o, xm, vh), link_b(U, mu, e, xmyp, vh));
    step_end(t);
    t = m3_dmul(t, link_b(U, mu, o, xm, vh));
    step_end(t);
    im_tr_j(r, m3_mul(own(nu), t), s);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; j++) {
    lds.part[k][0][j][lane] = q[j];
    lds.part[k][1][j][lane] = r[j];
  }
  __syncthreads();
  if (k > 3 || !active) return;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    // planes 01 02 03 12 13 23; 0: the first direction's share, 1: the second's
    const auto part = [&](int p, int d) { return lds.part[p][d][j][lane]; };
    q[j] = k == 0 ? part(0, 0) + part(1, 0) + part(2, 0)
         : k == 1 ? part(0, 1) + part(3, 0) + part(4, 0)
         : k == 2 ? part(1, 1) + part(3, 1) + part(5, 0)
                  : part(2, 1) + part(4, 1) + part(5, 1);
  }
  mom_add(P, k, e, i, vh, q);
}

// ---------------------------------------------------------------------------
// link update (hmc_u.F90:46-56): U <- exp(i step p.lambda) U, reunitarised
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(128) void k_hmc_u(double2 *__restrict__ U, const double *__restrict__ P, Geom g,
                                               double step) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int me = blockIdx.y, mu = me >> 1, e = me & 1;
  if (i >= g.vh) return;
  double h[8];
  const double *p = P + (size_t)(me * 8) * g.vh + i;
#pragma unroll
  for (int j = 0; j < 8; j++) h[j] = p[(size_t)j * g.vh] * step;
  M3 u = m3_mul(m3_expi(gellmann(h)), link(U, mu, e, i, g.vh));
  m3_reunitarize(u);
  store_link(U, mu, e, i, g.vh, u);
}

// 2 * sum_i log(prod_k stored B_kk) over one parity (clover_action.F90:40-56)
__global__ __launch_bounds__(kBlock) void k_clover_action(const double2 *__restrict__ Cb, int eo, int vh,
                                                          double *partials) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0.0;
  if (i < vh) {
    double d = 1.0;
    for (int J = 0; J < 2; J++)
      for (int w = 15; w < 18; w++) {
        double2 v = Cb[(size_t)(eo * 36 + J * 18 + w) * vh + i];
        d *= v.x * v.y;
      }
    s = log(d);
  }
  double vals[1] = {s};
  block_partials<1>(vals, partials);
}

struct FinTwice {
  double *out;
  __device__ void operator()(const double (&t)[1]) const { out[0] = 2.0 * t[0]; }
};

// ---------------------------------------------------------------------------
// host drivers
// ---------------------------------------------------------------------------
double *mom_scratch(Context *c, int *rc) {
  return static_cast<double *>(scratch(c, SLOT_MOM, sizeof(double) * 64 * (size_t)c->g.vh, rc));
}

// scratch for six Hermitian 3x3 matrices per site of one parity (H3)
static double *h_scratch(Context *c, int slot, int *rc) {
  return static_cast<double *>(scratch(c, slot, sizeof(double) * 54 * (size_t)c->g.vh, rc));
}

// dsf.F90:28-110 on device spinors a, b (even parity); P accumulates
int dsf_dev(Context *c, double *P, double step, double kappa, double csw_kappa, const double2 *a,
            const double2 *b) {
  const int vh = c->g.vh;
  int rc = 0;
  double2 *at = spinor_scratch(c, SLOT_FORCE0, &rc); HB_TRY(rc);
  double2 *bt = spinor_scratch(c, SLOT_FORCE1, &rc); HB_TRY(rc);
  double *H0 = h_scratch(c, SLOT_FORCE2, &rc); HB_TRY(rc);
  double *H1 = h_scratch(c, SLOT_FORCE3, &rc); HB_TRY(rc);
  const bool clov = csw_kappa != 0.0;
  if (clov) HB_CHECK(c->have_clover[HB_CLOVER_B], HB_E_STATE, "dsf: clover B field not present");
  if (kappa != 0.0) {
    // A~ = D_oe a, B~ = D_eo^+ b (dsf.F90:56-57), then A_oo^-1 by LDL^+ (clover_mult_b)
    DslashArgs<SF64> d1 = dslash_args64(c, 1, at, a);
    if (clov) d1.C = c->clov[HB_CLOVER_B];
    HB_TRY(launch_dslash(d1, false, clov ? EPI_SOLVE : EPI_PLAIN, c->stream));
    DslashArgs<SF64> d2 = dslash_args64(c, 1, bt, b);
    d2.C = d1.C;
    HB_TRY(launch_dslash(d2, true, clov ? EPI_SOLVE : EPI_PLAIN, c->stream));
  }
  const LinkGrid lg(c->g);
  const HopForce hop{a, b, at, bt, -step * 2.0 * kappa * kappa};
  // clover part (dsf.F90:103-109) on physical links; at kappa = 0 neither the
  // hopping part nor the odd sites' clover part is there and nothing reads at, bt
  const double s1 = -step * 2.0 * (csw_kappa / 8.0);
  const double s2 = s1 * kappa * kappa;
  if (s1 != 0.0)
    k_h_spinors<<<dim3(nblocks(vh), s2 != 0.0 ? 2 : 1), kBlock, 0, c->stream>>>(HSpinors{H0, b, a, s1},
                                                                               HSpinors{H1, bt, at, s2}, vh);
  if (hop.s != 0.0 || s1 != 0.0)
    k_clover_force<true><<<lg.grid, kLinkBlock, 0, c->stream>>>(P, c->gauge, c->g, lg.run, s1 != 0.0 ? H0 : nullptr,
                                                                s2 != 0.0 ? H1 : nullptr, hop);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

// the clover force of one parity's H field
static int clover_force_one(Context *c, double *P, int eo, const double *H) {
  const LinkGrid lg(c->g);
  k_clover_force<false><<<lg.grid, kLinkBlock, 0, c->stream>>>(P, c->gauge, c->g, lg.run, eo == 0 ? H : nullptr,
                                                               eo == 0 ? nullptr : H, HopForce{});
  HB_HIP(hipGetLastError());
  return HB_OK;
}

// clover_dsf (clover/clover_d.F90:78-106) of spinors b, a of parity eo with
// scale s, on the loaded (physical) links; P accumulates
int clover_dsf_dev(Context *c, double *P, int eo, const double2 *b, const double2 *a, double s) {
  if (s == 0.0) return HB_OK;
  int rc = 0;
  double *H = h_scratch(c, SLOT_FORCE2, &rc); HB_TRY(rc);
  const HSpinors h{H, b, a, s};
  k_h_spinors<<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(h, h, c->g.vh);
  return clover_force_one(c, P, eo, H);
}

// clover_dsd (clover/clover_d.F90:40-75) with the loaded LDL^+ field of parity eo
int clover_dsd_dev(Context *c, double *P, int eo, double s) {
  if (s == 0.0) return HB_OK;
  HB_CHECK(c->have_clover[HB_CLOVER_B], HB_E_STATE, "clover_dsd: clover B field not present");
  int rc = 0;
  double *H = h_scratch(c, SLOT_FORCE2, &rc); HB_TRY(rc);
  k_h_inverse<<<nblocks(c->g.vh), kBlock, 0, c->stream>>>(H, c->clov[HB_CLOVER_B], eo, c->g.vh, s);
  return clover_force_one(c, P, eo, H);
}

// dsd.F90:28-49 (clover_dsd on the odd sites)
int dsd_dev(Context *c, double *P, double step, double csw_kappa) {
  const double s = -step * 2.0 * (csw_kappa / 8.0);
  if (s != 0.0) HB_CHECK(c->have_clover[HB_CLOVER_B], HB_E_STATE, "dsd: clover B field not present");
  return clover_dsd_dev(c, P, 1, s);
}

// clover_action (clover/clover_action.F90:29-62) of parity eo of the LDL^+
// field Cb (device layout [2][36][vh])
int clover_action_parity_dev(Context *c, const double2 *Cb, int eo, double *res_d) {
  const int vh = c->g.vh;
  k_clover_action<<<nblocks(vh), kBlock, 0, c->stream>>>(Cb, eo, vh, c->red);
  k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(c->red, nblocks(vh), nullptr, FinTwice{res_d});
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int dsg_dev(Context *c, double *P, double step, double beta) {
  if (beta == 0.0) return HB_OK;
  const LinkGrid lg(c->g);
  k_gauge_force<<<lg.grid, kPlaneBlock, 0, c->stream>>>(P, c->gauge, c->g, lg.run, -step * beta / 3.0);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

int build_clover_dev(Context *c, double csw_kappa);

int hmc_u_dev(Context *c, const double *P, double step, double csw_kappa) {
  k_hmc_u<<<dim3(nblocks(c->g.vh, 128), 8), 128, 0, c->stream>>>(c->gauge, P, c->g, step);
  HB_HIP(hipGetLastError());
  c->gauge_version++;
  if (csw_kappa != 0.0) HB_TRY(build_clover_dev(c, csw_kappa));
  return HB_OK;
}

int clover_action_dev(Context *c, double *res_d) {
  HB_CHECK(c->have_clover[HB_CLOVER_B], HB_E_STATE, "clover_action: clover B field not present");
  const int vh = c->g.vh;
  k_clover_action<<<nblocks(vh), kBlock, 0, c->stream>>>(c->clov[HB_CLOVER_B], 1, vh, c->red);
  k_finalize<1><<<1, kFinThreads, 0, c->stream>>>(c->red, nblocks(vh), nullptr, FinTwice{res_d});
  HB_HIP(hipGetLastError());
  return HB_OK;
}

}  // namespace hb

using namespace hb;

extern "C" {

int hb_dsf_d(hb_context *ctx, double *p_d, double step, double kappa, double csw_kappa, const double *a_d,
             const double *b_d) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p_d && a_d && b_d, HB_E_ARG, "hb_dsf_d: null pointer");
  HB_HIP(hipSetDevice(c->device));
  return dsf_dev(c, p_d, step, kappa, csw_kappa, reinterpret_cast<const double2 *>(a_d),
                 reinterpret_cast<const double2 *>(b_d));
}

int hb_dsf(hb_context *ctx, double *p, int site_stride, double step, double kappa, double csw_kappa,
           const double *a, const double *b) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p && a && b, HB_E_ARG, "hb_dsf: null pointer");
  HB_CHECK(site_stride >= c->g.vh, HB_E_ARG, "hb_dsf: site_stride < volh");
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  double *P = mom_scratch(c, &rc); HB_TRY(rc);
  double2 *da = spinor_scratch(c, SLOT_X, &rc); HB_TRY(rc);
  double2 *db = spinor_scratch(c, SLOT_B, &rc); HB_TRY(rc);
  HB_TRY(gen_upload(c, P, p, site_stride));
  HB_TRY(spinor_upload(c, da, a));
  HB_TRY(spinor_upload(c, db, b));
  HB_TRY(dsf_dev(c, P, step, kappa, csw_kappa, da, db));
  return gen_download(c, p, P, site_stride);
}

int hb_dsd(hb_context *ctx, double *p, int site_stride, double step, double csw_kappa) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p && site_stride >= c->g.vh, HB_E_ARG, "hb_dsd: bad arguments");
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  double *P = mom_scratch(c, &rc); HB_TRY(rc);
  HB_TRY(gen_upload(c, P, p, site_stride));
  HB_TRY(dsd_dev(c, P, step, csw_kappa));
  return gen_download(c, p, P, site_stride);
}

int hb_dsg(hb_context *ctx, double *p, int site_stride, double step, double beta) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p && site_stride >= c->g.vh, HB_E_ARG, "hb_dsg: bad arguments");
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  double *P = mom_scratch(c, &rc); HB_TRY(rc);
  HB_TRY(gen_upload(c, P, p, site_stride));
  HB_TRY(dsg_dev(c, P, step, beta));
  return gen_download(c, p, P, site_stride);
}

int hb_hmc_u(hb_context *ctx, const double *p, int site_stride, double step, double csw_kappa) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p && site_stride >= c->g.vh, HB_E_ARG, "hb_hmc_u: bad arguments");
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  double *P = mom_scratch(c, &rc); HB_TRY(rc);
  HB_TRY(gen_upload(c, P, p, site_stride));
  HB_TRY(hmc_u_dev(c, P, step, csw_kappa));
  HB_HIP(hipStreamSynchronize(c->stream));
  return HB_OK;
}

int hb_hmc_u_d(hb_context *ctx, const double *p_d, double step, double csw_kappa) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p_d, HB_E_ARG, "hb_hmc_u_d: null pointer");
  HB_HIP(hipSetDevice(c->device));
  return hmc_u_dev(c, p_d, step, csw_kappa);
}

int hb_dsd_d(hb_context *ctx, double *p_d, double step, double csw_kappa) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p_d, HB_E_ARG, "hb_dsd_d: null pointer");
  HB_HIP(hipSetDevice(c->device));
  return dsd_dev(c, p_d, step, csw_kappa);
}

int hb_dsg_d(hb_context *ctx, double *p_d, double step, double beta) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(p_d, HB_E_ARG, "hb_dsg_d: null pointer");
  HB_HIP(hipSetDevice(c->device));
  return dsg_dev(c, p_d, step, beta);
}

int hb_clover_action(hb_context *ctx, double *s_det) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(s_det, HB_E_ARG, "hb_clover_action: null pointer");
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  double *r = static_cast<double *>(scratch(c, SLOT_STATE, sizeof(CgState), &rc)); HB_TRY(rc);
  HB_TRY(clover_action_dev(c, r));
  HB_HIP(hipMemcpyAsync(s_det, r, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HB_HIP(hipStreamSynchronize(c->stream));
  return HB_OK;
}

int hb_gauge_backup(hb_context *ctx, int slot) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(slot >= 0 && slot < kGaugeBackups, HB_E_ARG, "hb_gauge_backup: slot %d (0..%d)", slot, kGaugeBackups - 1);
  HB_HIP(hipSetDevice(c->device));
  int rc = 0;
  void *dst = scratch(c, SLOT_BACKUP + slot, sizeof(double2) * 72 * (size_t)c->g.vh, &rc); HB_TRY(rc);
  HB_HIP(hipMemcpyAsync(dst, c->gauge, sizeof(double2) * 72 * (size_t)c->g.vh, hipMemcpyDeviceToDevice, c->stream));
  return HB_OK;
}

int hb_gauge_restore(hb_context *ctx, int slot) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_TRY(check_ready(c));
  HB_CHECK(slot >= 0 && slot < kGaugeBackups, HB_E_ARG, "hb_gauge_restore: slot %d (0..%d)", slot, kGaugeBackups - 1);
  HB_CHECK((int)c->scratch.size() > SLOT_BACKUP + slot && c->scratch[SLOT_BACKUP + slot].p, HB_E_STATE,
           "hb_gauge_restore: slot %d never backed up", slot);
  HB_HIP(hipSetDevice(c->device));
  HB_HIP(hipMemcpyAsync(c->gauge, c->scratch[SLOT_BACKUP + slot].p, sizeof(double2) * 72 * (size_t)c->g.vh,
                        hipMemcpyDeviceToDevice, c->stream));
  c->gauge_version++;
  return HB_OK;
}

}  // extern "C"
