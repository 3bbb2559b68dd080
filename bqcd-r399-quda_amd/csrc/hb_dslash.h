// hb_dslash.h - launch interface of the fused hopping-matrix kernels.
#pragma once

#include "hb_blas.h"

namespace hb {

enum { EPI_PLAIN = 0, EPI_CLINV = 1, EPI_MTIL = 2, EPI_MTDOT = 3, EPI_SOLVE = 4 };

// S: spinor storage; G: link and clover storage (same arithmetic type as S)
template <class S, class G = S> struct DslashArgs {
  Geom g;
  int out_parity;
  SpinorPtr<S> out;
  SpinorPtr<S> in;
  const typename G::ST *U;   // links [4][2][9][vh]
  const typename G::ST *C;   // clover field for the epilogue (A^-1 for CLINV, A for MTIL, LDL^+ for SOLVE), or null
  const float *Cn;           // 16-bit clover: (scale, diagonal offset) per site and block
  SpinorPtr<S> x0;           // MTIL: the vector the clover term acts on
  SpinorPtr<S> dotv;         // MTDOT: Re<dotv, out>
  double mkappa2;            // -kappa^2
  double rho;
  double *partials;          // MTDOT: per-workgroup partial sums (dslash_grid doubles)
  const int *skip;           // if non-null and *skip != 0 the launch does nothing
};

// Load policy of the links and clover words, which a kernel reads once: kept
// in the caches while the operator and the vectors of a solve are up to 1.4 to
// 1.8 times as large as the 256 MB last-level cache, streamed past them (so that
// the neighbour spinors stay) beyond.  The lines in MiB of that working set, with
// us streamed / kept on either side (sites per parity):
//   M~^+M~ in FP64, 18-real links 340: 104 k (332 MiB) 175 / 171, 112 k (359) 183 / 188;
//       D alone, which reads no clover words, 360: 112 k 34.1 / 32.0, 120 k 35.7 / 36.0
//   CG iteration, FP64 372: 120 k (341) 215 / 205, 128 k (363) 225 / 216, 141 k (400) 254 / 288
//   FP32 450: 249 k (364) 294 / 271, 304 k (446) 345 / 334, 332 k (486) 390 / 392; blocks of
//       two 219 k (441) 423 / 416, 249 k (501) 480 / 485, of four 141 k (438) 561 / 544,
//       200 k (623) 776 / 785
//   16-bit 434: 470 k (389) 335 / 319, 524 k (434) 336 / 331, 655 k (543) 423 / 431; blocks 360:
//       two 304 k (355) 361 / 360, 359 k (420) 441 / 444, four 200 k (369) 478 / 474,
//       249 k (459) 578 / 580
//   FP32 spinors, 16-bit links and clover 385: 359 k (373) 321 / 311, 432 k (448) 386 / 390
template <class S, class G> constexpr size_t resident_bytes(int nr, bool clover) {
  const size_t mib = std::is_same<S, SF64>::value   ? (G::kRecon ? 372 : clover ? 340 : 360)
                     : std::is_same<S, SF16>::value ? (nr == 1 ? 434 : 360)
                     : std::is_same<G, SF16>::value ? 385 : 450;
  return mib << 20;
}
template <class S, class G> constexpr size_t solve_bytes_per_site(int nr = 1) {
  const size_t link = std::is_same<G, SF16>::value ? 24 : G::kRecon ? 6 * G::kBytes : 9 * G::kBytes;
  const size_t clov = std::is_same<G, SF16>::value ? 2 * kClov16 : 36 * G::kBytes;
  const size_t spin = 12 * S::kBytes + (S::kNorm ? 4 : 0);
  return 8 * link + 2 * clov + (5 * spin + 96) * nr;  // p, r, q, t, y and the FP32 increment
}
template <class S, class G> inline int operator_policy(int vh, int nr = 1, bool clover = true) {
  return solve_bytes_per_site<S, G>(nr) * (size_t)vh <= resident_bytes<S, G>(nr, clover) ? 0 : kNT;
}
// the largest lattice (sites per parity) whose operator is kept
template <class S, class G> constexpr int kept_sites(bool clover) {
  return (int)(resident_bytes<S, G>(1, clover) / solve_bytes_per_site<S, G>());
}

// Waves that share a site (1: k_dslash, else k_dslash_split).  us per CG
// iteration at 1 / 2 / 4 waves:
//   FP64    8^4 (2 k sites per parity) 58.9 / 47.1 / 45.0, 12^3x24 (21 k)
//           80.3 / 61.5 / 58.4, 16^4 (33 k) 85.4 / 69.0 / 69.2,
//           16x16x18x18 (41 k) 91.3 / 79.4 / 89.8, 16^3x32 (66 k) 117 / 112 / 112,
//           24x20x12x36 (104 k) 184 / 178, 20^3x40 (160 k) 273 / 274, 24^3x48
//           (332 k) 570 / 580 (the one wave in workgroups of 64 sites);
//           M~^+M~ with 18-real links 41 k 66.8 / 63.4 / 68.8, 50 k 74.2 / 80.2 / 82.1
//   FP32    12^3x24 70.7 / 58.7 / 57.6, 16^4 69.5 / 61.5 / 59.4, 50 k 77.0 / 71.1 /
//           72.2, 24^3x48 (332 k) 365 / 356 / 358, 32^3x64 1010 / 1056 / 1067
//   16-bit  12^3x24 60.9 / 55.4 / 52.2, 50 k 62.9 / 58.7 / 60.6, 24^3x48
//           207 / 200 / 214, 32^3x64 522 / 548 / 580
//   around the line of both, at 1 / 2: FP32 470 k 547 / 547, 524 k 559 / 573, 590 k 653 / 668,
//           655 k 717 / 735; 16-bit 334 / 334, 329 / 336, 394 / 400, 424 / 432
// Eight waves (one hop each) were slower than four from 4 k sites on.
constexpr int kFourWaveSites = 1 << 15;
template <class S, class G> constexpr int two_wave_sites() {
  return !std::is_same<S, SF64>::value ? 1 << 19 : G::kRecon ? 1 << 17 : 3 << 14;
}
template <class S, class G> inline int split_waves(int vh) {
  return vh <= kFourWaveSites ? 4 : vh <= two_wave_sites<S, G>() ? 2 : 1;
}

// Sites per workgroup.  One wave per site in FP64 runs two workgroups of 256
// per CU: where that is a few rounds of the chip, workgroups of one wave leave
// less of it idle in the last one.  256 / 64 sites, us, FP64 CG iteration and
// M~^+M~ with 18-real links: 24x20x12x36 (104 k sites per parity, one round) 184 /
// 183 and 170 / 176, 20^3x40 (160 k) 288 / 276 and 265 / 257, 24^3x48 (332 k) 592 /
// 574 and 569 / 545, 28x28x28x36 (395 k) 689 / 666 and 627 / 600, 32x32x32x28 (459 k) 771 /
// 768 and 725 / 732, 28x28x30x40 (470 k) 834 / 826 and 807 / 792, 32^4 (524 k) 854 / 856 and
// 810 / 805, 32^3x64 (1049 k) 1693 / 1699 and 1621 / 1624.  FP32 and 16-bit fields, at higher occupancy: 354 / 352 and 196 / 194 at 24^3x48, 998 / 1023 and
// 503 / 507 at 32^3x64.
template <class S, class G> inline int dslash_tile(int vh) {
  if (split_waves<S, G>(vh) > 1) return 64;
  return std::is_same<S, SF64>::value && vh > (1 << 17) && vh <= (1 << 19) ? 64 : kBlock;
}
// workgroups of a launch, each of which leaves one partial sum (EPI_MTDOT)
template <class S, class G> inline int dslash_grid(int vh) {
  return nblocks(vh, dslash_tile<S, G>(vh));
}

template <class S, class G> int launch_dslash(const DslashArgs<S, G> &a, bool dag, int epi, hipStream_t st);

}  // namespace hb
