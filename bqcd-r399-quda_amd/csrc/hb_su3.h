// hb_su3.h - 3x3 complex matrices in registers (FP64) for the clover build,
// forces, link update and gauge generation kernels.
#pragma once

#include <algorithm>

#include "hb_kernels.h"

namespace hb {

struct M3 {
  double2 m[9];  // row-major: m[3*r + c]
};

__device__ __forceinline__ M3 m3_zero() {
  M3 r;
#pragma unroll
  for (int k = 0; k < 9; k++) r.m[k] = make_double2(0.0, 0.0);
  return r;
}
// s += a' b' with a' = conj(a) if CA, b' = conj(b) if CB: four chained FMAs
// (the force, clover and link-update kernels are bound by FP64 issue; the
// sign flips are free operand modifiers)
template <bool CA, bool CB>
__device__ __forceinline__ void cfma3(double2 &s, double2 a, double2 b) {
  const double ay = CA ? -a.y : a.y, by = CB ? -b.y : b.y;
  s.x = fma(a.x, b.x, s.x);
  s.x = fma(-ay, by, s.x);
  s.y = fma(a.x, by, s.y);
  s.y = fma(ay, b.x, s.y);
}
// Re(a' b') only
template <bool CA, bool CB>
__device__ __forceinline__ double cfma3_re(double s, double2 a, double2 b) {
  const double ay = CA ? -a.y : a.y, by = CB ? -b.y : b.y;
  return fma(-ay, by, fma(a.x, b.x, s));
}

// element (i, j) of a b (MODE 0), a^+ b (MODE 1) or a b^+ (MODE 2)
template <int MODE>
__device__ __forceinline__ double2 m3_elem(const M3 &a, const M3 &b, int i, int j) {
  double2 s = make_double2(0.0, 0.0);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    if constexpr (MODE == 0) cfma3<false, false>(s, a.m[3 * i + k], b.m[3 * k + j]);
    else if constexpr (MODE == 1) cfma3<true, false>(s, a.m[3 * k + i], b.m[3 * k + j]);
    else cfma3<false, true>(s, a.m[3 * i + k], b.m[3 * j + k]);
  }
  return s;
}
template <int MODE>
__device__ __forceinline__ double m3_elem_re(const M3 &a, const M3 &b, int i, int j) {
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    if constexpr (MODE == 0) s = cfma3_re<false, false>(s, a.m[3 * i + k], b.m[3 * k + j]);
    else if constexpr (MODE == 1) s = cfma3_re<true, false>(s, a.m[3 * k + i], b.m[3 * k + j]);
    else s = cfma3_re<false, true>(s, a.m[3 * i + k], b.m[3 * j + k]);
  }
  return s;
}
template <int MODE> __device__ __forceinline__ M3 m3_prod(const M3 &a, const M3 &b) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) r.m[3 * i + j] = m3_elem<MODE>(a, b, i, j);
  return r;
}
__device__ __forceinline__ M3 m3_mul(const M3 &a, const M3 &b) { return m3_prod<0>(a, b); }
// a^+ b
__device__ __forceinline__ M3 m3_dmul(const M3 &a, const M3 &b) { return m3_prod<1>(a, b); }
// a b^+
__device__ __forceinline__ M3 m3_muld(const M3 &a, const M3 &b) { return m3_prod<2>(a, b); }
__device__ __forceinline__ void m3_acc(M3 &a, const M3 &b) {
#pragma unroll
  for (int k = 0; k < 9; k++) a.m[k] = cadd(a.m[k], b.m[k]);
}
__device__ __forceinline__ void m3_scale(M3 &a, double s) {
#pragma unroll
  for (int k = 0; k < 9; k++) a.m[k] = cscale<double2>(s, a.m[k]);
}
__device__ __forceinline__ double m3_retr(const M3 &a) { return a.m[0].x + a.m[4].x + a.m[8].x; }

// link U_mu(x) of parity eo at site i (physical links, SoA gauge)
__device__ __forceinline__ M3 link(const double2 *__restrict__ U, int mu, int eo, int i, int vh) {
  M3 r;
  const double2 *b = U + (size_t)((mu * 2 + eo) * 9) * vh + i;
#pragma unroll
  for (int k = 0; k < 9; k++) r.m[k] = b[(size_t)k * vh];
  return r;
}
// the same through a buffer resource over the (mu, eo) slab (mu, eo
// wave-uniform): one 32-bit offset register per matrix instead of nine 64-bit
// addresses; slab offsets stay below 2^32 bytes up to vh = 2^32 / 144
__device__ __forceinline__ M3 link_b(const double2 *__restrict__ U, int mu, int eo, int i, int vh) {
  const uint32_t plane = (uint32_t)vh * 16u;
  const rsrc_t r = make_rsrc(U + (size_t)((mu * 2 + eo) * 9) * vh, plane * 9u);
  const uint32_t vo = (uint32_t)i * 16u;
  M3 m;
#pragma unroll
  for (int k = 0; k < 9; k++) m.m[k] = bld_f64x2(r, vo, plane * (uint32_t)k);
  return m;
}
__device__ __forceinline__ void store_link(double2 *__restrict__ U, int mu, int eo, int i, int vh,
                                           const M3 &v) {
  double2 *b = U + (size_t)((mu * 2 + eo) * 9) * vh + i;
#pragma unroll
  for (int k = 0; k < 9; k++) b[(size_t)k * vh] = v.m[k];
}

// an index the compiler cannot prove equal to its argument: a matrix loaded
// again through it is a fresh load, not a register kept live since the first
__device__ __forceinline__ int fresh(int i) {
  asm volatile("" : "+v"(i));
  return i;
}

// Ends a step of a kernel: the matrix is complete in registers here, and no
// load of a later step is issued before.
__device__ __forceinline__ void pin(M3 &m) {
#pragma unroll
  for (int k = 0; k < 9; k++) asm volatile("" : "+v"(m.m[k].x), "+v"(m.m[k].y));
}
__device__ __forceinline__ void step_end(M3 &m) {
  pin(m);
  __builtin_amdgcn_sched_barrier(0);
}

// neighbour index (parity of the result is 1 - eo for a single step)
__device__ __forceinline__ int nb(const Geom &g, int x, int y, int z, int t, int mu, int d) {
  int c[4] = {x, y, z, t};
  c[mu] += d;
  if (c[mu] >= g.L[mu]) c[mu] -= g.L[mu];
  if (c[mu] < 0) c[mu] += g.L[mu];
  return site_index(g, c[0], c[1], c[2], c[3]);
}
__device__ __forceinline__ int nb2(const Geom &g, int x, int y, int z, int t, int mu, int dm,
                                   int nu, int dn) {
  int c[4] = {x, y, z, t};
  c[mu] += dm;
  c[nu] += dn;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if (c[k] >= g.L[k]) c[k] -= g.L[k];
    if (c[k] < 0) c[k] += g.L[k];
  }
  return site_index(g, c[0], c[1], c[2], c[3]);
}

// Gram-Schmidt of the first two columns, third column = conj(cross product)
// (the reunitarisation of su3.F90:313-365)
__device__ __forceinline__ void m3_reunitarize(M3 &u) {
  double len = 0.0;
#pragma unroll
  for (int r = 0; r < 3; r++) len += u.m[3 * r].x * u.m[3 * r].x + u.m[3 * r].y * u.m[3 * r].y;
  len = sqrt(len);
#pragma unroll
  for (int r = 0; r < 3; r++) u.m[3 * r] = make_double2(u.m[3 * r].x / len, u.m[3 * r].y / len);
  double2 f = make_double2(0.0, 0.0);
#pragma unroll
  for (int r = 0; r < 3; r++) cfmac(f, u.m[3 * r], u.m[3 * r + 1]);  // sum conj(u_r0) u_r1
#pragma unroll
  for (int r = 0; r < 3; r++) u.m[3 * r + 1] = csub(u.m[3 * r + 1], cmul(f, u.m[3 * r]));
  len = 0.0;
#pragma unroll
  for (int r = 0; r < 3; r++)
    len += u.m[3 * r + 1].x * u.m[3 * r + 1].x + u.m[3 * r + 1].y * u.m[3 * r + 1].y;
  len = sqrt(len);
#pragma unroll
  for (int r = 0; r < 3; r++) u.m[3 * r + 1] = make_double2(u.m[3 * r + 1].x / len, u.m[3 * r + 1].y / len);
  u.m[2] = cconj(csub(cmul(u.m[3], u.m[7]), cmul(u.m[6], u.m[4])));
  u.m[5] = cconj(csub(cmul(u.m[6], u.m[1]), cmul(u.m[0], u.m[7])));
  u.m[8] = cconj(csub(cmul(u.m[0], u.m[4]), cmul(u.m[3], u.m[1])));
}

// H = sum_j h_j lambda_j (Gell-Mann basis of su3.F90:196-233)
__device__ __forceinline__ M3 gellmann(const double (&h)[8]) {
  const double s3 = 0.57735026918962576;  // 1/sqrt(3)
  M3 H;
  H.m[0] = make_double2(h[2] + s3 * h[7], 0.0);
  H.m[4] = make_double2(-h[2] + s3 * h[7], 0.0);
  H.m[8] = make_double2(-2.0 * s3 * h[7], 0.0);
  H.m[1] = make_double2(h[0], -h[1]);
  H.m[3] = make_double2(h[0], h[1]);
  H.m[2] = make_double2(h[3], -h[4]);
  H.m[6] = make_double2(h[3], h[4]);
  H.m[5] = make_double2(h[5], -h[6]);
  H.m[7] = make_double2(h[5], h[6]);
  return H;
}

// exp(i H) for a Hermitian traceless H (the exponential map of gen2u,
// su3.F90:28-193, by a different method): Taylor series with scaling and
// squaring.  With X = H / 2^sq, X^3 = c0 + c1 X (Cayley-Hamilton, c0 = det X,
// c1 = Tr X^2 / 2) makes every power a_n + b_n X + c_n X^2, so that the series
// runs over three real numbers per term and one matrix product, X^2, is left;
// summed as matrices its 18 products kept the link update on FP64 issue
// (24x20x12x36: 108 us, now 48 us or 6 TB/s).  sq is chosen for |X| <= 1, where twenty
// terms leave less than 1e-19.
__device__ __forceinline__ M3 m3_expi(const M3 &H) {
  double nrm = 0.0;
#pragma unroll
  for (int k = 0; k < 9; k++) nrm += fabs(H.m[k].x) + fabs(H.m[k].y);
  int sq = 0;
  while (nrm > 1.0 && sq < 60) { nrm *= 0.5; sq++; }
  const double sc = ldexp(1.0, -sq);
  const double d0 = sc * H.m[0].x, d1 = sc * H.m[4].x, d2 = sc * H.m[8].x;
  const double2 p = cscale<double2>(sc, H.m[1]), q = cscale<double2>(sc, H.m[2]), r = cscale<double2>(sc, H.m[5]);
  const double pp = p.x * p.x + p.y * p.y, qq = q.x * q.x + q.y * q.y, rr = r.x * r.x + r.y * r.y;
  // X^2: diagonal s0, s1, s2, upper triangle u (01), v (02), w (12)
  const double s0 = d0 * d0 + pp + qq, s1 = d1 * d1 + pp + rr, s2 = d2 * d2 + qq + rr;
  double2 u = cscale<double2>(d0 + d1, p), v = cscale<double2>(d0 + d2, q), w = cscale<double2>(d1 + d2, r);
  cfma3<false, true>(u, q, r);   // X02 X21 = q conj(r)
  cfma3<false, false>(v, p, r);  // X01 X12
  cfma3<true, false>(w, p, q);   // X10 X02
  const double2 pr = cmul(p, r);
  const double c1 = 0.5 * (s0 + s1 + s2);
  const double c0 = d0 * d1 * d2 + 2.0 * (pr.x * q.x + pr.y * q.y) - d0 * rr - d1 * qq - d2 * pp;
  // sum_n i^n (a_n, b_n, c_n) / n!, real and imaginary part
  double a = 1.0, b = 0.0, c = 0.0;
  double f0[2] = {1.0, 0.0}, f1[2] = {0.0, 0.0}, f2[2] = {0.0, 0.0};
#pragma unroll
  for (int n = 1; n <= 20; n++) {
    const double in = 1.0 / n, na = c0 * c * in, nb = fma(c1, c, a) * in;
    c = b * in;
    a = na;
    b = nb;
    const double sg = (n & 2) ? -1.0 : 1.0;
    f0[n & 1] = fma(sg, a, f0[n & 1]);
    f1[n & 1] = fma(sg, b, f1[n & 1]);
    f2[n & 1] = fma(sg, c, f2[n & 1]);
  }
  const double2 g0 = make_double2(f0[0], f0[1]), g1 = make_double2(f1[0], f1[1]), g2 = make_double2(f2[0], f2[1]);
  M3 R;
  const auto diag = [&](double x, double y) {
    return make_double2(fma(g2.x, y, fma(g1.x, x, g0.x)), fma(g2.y, y, fma(g1.y, x, g0.y)));
  };
  R.m[0] = diag(d0, s0);
  R.m[4] = diag(d1, s1);
  R.m[8] = diag(d2, s2);
  const auto off = [&](double2 x, double2 y) {
    double2 z = cmul(g1, x);
    cfma3<false, false>(z, g2, y);
    return z;
  };
  R.m[1] = off(p, u);
  R.m[3] = off(cconj(p), cconj(u));
  R.m[2] = off(q, v);
  R.m[6] = off(cconj(q), cconj(v));
  R.m[5] = off(r, w);
  R.m[7] = off(cconj(r), cconj(w));
  for (int s = 0; s < sq; s++) R = m3_mul(R, R);
  return R;
}

// p_j += s * Im Tr(lambda_j v)  (su3.F90:196-213)
__device__ __forceinline__ void im_tr_j(double (&p)[8], const M3 &v, double s) {
  const double is3 = 0.57735026918962576;
  p[0] += s * (v.m[1].y + v.m[3].y);
  p[1] += s * (v.m[1].x - v.m[3].x);
  p[2] += s * (v.m[0].y - v.m[4].y);
  p[3] += s * (v.m[2].y + v.m[6].y);
  p[4] += s * (v.m[2].x - v.m[6].x);
  p[5] += s * (v.m[5].y + v.m[7].y);
  p[6] += s * (v.m[5].x - v.m[7].x);
  p[7] += s * (v.m[0].y + v.m[4].y - 2.0 * v.m[8].y) * is3;
}

// p_j += s * Re Tr(lambda_j a b) (MODE 0) or Re Tr(lambda_j a b^+) (MODE 2),
// the elements of the product formed one at a time (the diagonal only in its
// real part) instead of as a matrix: the clover force evaluates 24 such terms
// per link and plane and is bound by registers and FP64 issue
template <int MODE>
__device__ __forceinline__ void re_tr_j_prod(double (&p)[8], const M3 &a, const M3 &b, double s) {
  const double is3 = 0.57735026918962576;
  {
    const double d0 = m3_elem_re<MODE>(a, b, 0, 0), d1 = m3_elem_re<MODE>(a, b, 1, 1);
    const double d2 = m3_elem_re<MODE>(a, b, 2, 2);
    p[2] += s * (d0 - d1);
    p[7] += s * (d0 + d1 - 2.0 * d2) * is3;
  }
  {
    const double2 x01 = m3_elem<MODE>(a, b, 0, 1), x10 = m3_elem<MODE>(a, b, 1, 0);
    p[0] += s * (x01.x + x10.x);
    p[1] += s * (x10.y - x01.y);
  }
  {
    const double2 x02 = m3_elem<MODE>(a, b, 0, 2), x20 = m3_elem<MODE>(a, b, 2, 0);
    p[3] += s * (x02.x + x20.x);
    p[4] += s * (x20.y - x02.y);
  }
  {
    const double2 x12 = m3_elem<MODE>(a, b, 1, 2), x21 = m3_elem<MODE>(a, b, 2, 1);
    p[5] += s * (x12.x + x21.x);
    p[6] += s * (x21.y - x12.y);
  }
}

// p_j += s * Re Tr(lambda_j v)  (su3.F90:216-233)
__device__ __forceinline__ void re_tr_j(double (&p)[8], const M3 &v, double s) {
  const double is3 = 0.57735026918962576;
  p[0] += s * (v.m[1].x + v.m[3].x);
  p[1] += s * (v.m[3].y - v.m[1].y);
  p[2] += s * (v.m[0].x - v.m[4].x);
  p[3] += s * (v.m[2].x + v.m[6].x);
  p[4] += s * (v.m[6].y - v.m[2].y);
  p[5] += s * (v.m[5].x + v.m[7].x);
  p[6] += s * (v.m[7].y - v.m[5].y);
  p[7] += s * (v.m[0].x + v.m[4].x - 2.0 * v.m[8].x) * is3;
}

// counter-based random numbers: splitmix64 of (seed, stream, index)
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}
struct Rng {
  uint64_t s;
  __device__ __forceinline__ Rng(uint64_t seed, uint64_t id) : s(splitmix64(seed ^ splitmix64(id))) {}
  __device__ __forceinline__ double uniform() {  // (0, 1]
    s = splitmix64(s);
    return ((double)(s >> 11) + 1.0) * (1.0 / 9007199254740992.0);
  }
  __device__ __forceinline__ void gauss2(double &a, double &b) {
    double r = sqrt(-2.0 * log(uniform()));
    double ph = 6.2831853071795862 * uniform();
    a = r * cos(ph);
    b = r * sin(ph);
  }
};

// Hermitian 3x3 matrices.  A field of one parity holds six of them per site
// (one per plane mu < nu): nine real planes of vh sites each, addressed as the
// double2 planes H01, H02, H12, (H00, H11) and the double plane H22.
struct H3 {
  double2 o[3];  // H01, H02, H12
  double d[3];
};

__device__ __forceinline__ void store_h(double *__restrict__ F, int k, int i, int vh, const H3 &h) {
  double *b = F + (size_t)k * 9 * vh;
  double2 *c = reinterpret_cast<double2 *>(b) + i;
  c[0] = h.o[0];
  c[vh] = h.o[1];
  c[2 * (size_t)vh] = h.o[2];
  c[3 * (size_t)vh] = make_double2(h.d[0], h.d[1]);
  b[8 * (size_t)vh + i] = h.d[2];
}
__device__ __forceinline__ H3 load_h(const double *__restrict__ F, int k, int i, int vh) {
  const uint32_t plane = (uint32_t)vh * 16u;
  const rsrc_t r = make_rsrc(F + (size_t)k * 9 * vh, (uint32_t)vh * 72u);
  const uint32_t vo = (uint32_t)i * 16u;
  H3 h;
#pragma unroll
  for (int q = 0; q < 3; q++) h.o[q] = bld_f64x2(r, vo, plane * (uint32_t)q);
  const double2 d = bld_f64x2(r, vo, plane * 3u);
  h.d[0] = d.x;
  h.d[1] = d.y;
  h.d[2] = __builtin_bit_cast(double, bld_u32x2(r, (uint32_t)i * 8u, plane * 4u));
  return h;
}

// Grid of the force and clover kernels: a workgroup holds the four directions of 64
// consecutive sites of one parity (one wave per direction or plane), its neighbour in
// the launch the other parity of the same sites.  All links of a neighbourhood
// are then read at about the same time, instead of by eight passes over the
// lattice, one per (direction, parity).  The XCDs share out every time slice
// in contiguous runs of `run` workgroups, so that the slices t and t +- 1 that
// all of them read stay in the last-level cache.  At 32^3x64 the gauge force
// takes 3.39 ms in eight passes, 1.78 ms with one contiguous eighth of the
// lattice per XCD, and 1.73 ms (1.54 ms in a single launch) with shared slices.
constexpr int kLinkBlock = 256;
struct LinkGrid {
  int grid, run;
  explicit LinkGrid(const Geom &g)
      : grid(2 * nblocks(g.vh, 64)), run(std::max(1, nblocks(g.vh / g.L[3], 256))) {}
};
__device__ __forceinline__ bool link_slot(const Geom &g, int run, int &mu, int &e, int &i) {
  int b = blockIdx.x;
  if (b < (int)gridDim.x / (8 * run) * (8 * run)) {
    const int x = b & 7, k = b >> 3;  // XCD (see xcd_block) and the workgroup's place in it
    b = k / run * (8 * run) + x * run + k % run;
  }
  mu = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  e = b & 1;
  i = (b >> 1) * 64 + ((int)threadIdx.x & 63);
  return i < g.vh;
}

}  // namespace hb
