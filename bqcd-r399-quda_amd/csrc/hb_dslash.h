// hb_dslash.h - launch interface of the fused hopping-matrix kernels.
#pragma once

#include "hb_blas.h"

namespace hb {

enum { EPI_PLAIN = 0, EPI_CLINV = 1, EPI_MTIL = 2, EPI_MTDOT = 3 };

// S: spinor storage; G: link and clover storage (same arithmetic type as S)
template <class S, class G = S> struct DslashArgs {
  Geom g;
  int out_parity;
  SpinorPtr<S> out;
  SpinorPtr<S> in;
  const typename G::ST *U;   // links [4][2][9][vh]
  const typename G::ST *C;   // clover field for the epilogue (A^-1 for CLINV, A for MTIL), or null
  const float *Cn;           // 16-bit clover: (scale, diagonal offset) per site and block
  SpinorPtr<S> x0;           // MTIL: the vector the clover term acts on
  SpinorPtr<S> dotv;         // MTDOT: Re<dotv, out>
  double mkappa2;            // -kappa^2
  double rho;
  double *dot_out;           // MTDOT result (device)
  double *partials;          // MTDOT per-block partial sums (gridDim doubles)
  const int *skip;           // if non-null and *skip != 0 the launch does nothing
};

// Load policy of the links and clover words, which a kernel reads once: kept
// in the caches while the operator and the vectors of a solve fit the 256 MB
// last-level cache, streamed past them (so that the neighbour spinors stay)
// when they do not.  CG iteration streamed / kept:
//   FP64    12^3x24 (50 MB) 96.6 / 79.5 us, 16^3x32 (157 MB) 130 / 116 us,
//           24^3x48 (796 MB) 605 / 666 us
//   FP32    14x20x12x30 (63 MB) 88.1 / 77.5 us, 24^3x48 (414 MB) 363 / 373 us
//   16-bit  24^3x48 (235 MB) 218 / 208 us, 32^3x64 (742 MB) 522 / 584 us
//           two right-hand sides at 24^3x48 (353 MB) 340 / 352 us
constexpr size_t kResidentBytes = (size_t)1 << 28;
template <class S, class G> constexpr size_t solve_bytes_per_site(int nr = 1) {
  const size_t link = std::is_same<G, SF16>::value ? 24 : G::kRecon ? 6 * G::kBytes : 9 * G::kBytes;
  const size_t clov = std::is_same<G, SF16>::value ? 2 * kClov16 : 36 * G::kBytes;
  const size_t spin = 12 * S::kBytes + (S::kNorm ? 4 : 0);
  return 8 * link + 2 * clov + (5 * spin + 96) * nr;  // p, r, q, t, y and the FP32 increment
}
template <class S, class G> inline int operator_policy(int vh, int nr = 1) {
  return solve_bytes_per_site<S, G>(nr) * (size_t)vh <= kResidentBytes ? 0 : kNT;
}

template <class S, class G> int launch_dslash(const DslashArgs<S, G> &a, bool dag, int epi, hipStream_t st);

}  // namespace hb
