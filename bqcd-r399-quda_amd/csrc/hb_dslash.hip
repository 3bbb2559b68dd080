// hb_dslash.hip - fused even-odd clover-Wilson hopping matrix.
//
// One thread per output site.  Each thread gathers the 8 neighbour spinors
// (coalesced: neighbours of consecutive sites are consecutive in the SoA
// planes), projects them to half spinors in registers, multiplies by the 8
// links and reconstructs -- the whole of d/D21.F90:29-76 (projection, the
// four direction passes and the out read-modify-write) in a single pass that
// reads each operand once and writes the result once.  Periodic wrap and the
// antiperiodic sign are computed on the device from the site coordinates.
//
// Epilogues fuse the operator algebra of m_tilde.F90:43-114 into the write:
//   EPI_PLAIN  out = D in
//   EPI_CLINV  out = A^-1 (D in)                      (clover_mult_ao on conf%i)
//   EPI_SOLVE  the same by LDL^+ substitution             (clover_mult_b on conf%b; FP64)
//   EPI_MTIL   out = A x0 - kappa^2 (D in) + rho x0   (clover_mult_a + sc_xpby + sc_axpy)
//   EPI_MTDOT  EPI_MTIL and the partial sums of Re<v, out> (sc_dot) per workgroup
#include "hb_dslash.h"
#include "hb_hop.h"

namespace hb {

template <class S, class G, bool DAG, int EPI, int POL>
__global__ __launch_bounds__(kBlock) void k_dslash(DslashArgs<S, G> a) {
  using V = typename S::V;
  using A = typename S::A;
  const Geom g = a.g;
  const int vh = g.vh;
  if (a.skip && *a.skip) return;
  const int i = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  V acc[12];
#pragma unroll
  for (int k = 0; k < 12; k++) acc[k] = cmk<V>((A)0, (A)0);
  const int e = a.out_parity;
  const bool active = i < vh;
  if (active) {
    int xc[4];
    site_coords(g, e, i, xc[0], xc[1], xc[2], xc[3]);
    const SpinorView<S> in(a.in, vh);
    if constexpr (HB_WAVE_SHARE && std::is_same<S, SF16>::value) {
      uint32_t w[13];
      in.load_words(w, i);
      const WaveView16 wv{in, w, i - (int)(threadIdx.x & 63), g.L[0] / 2 <= 32};
      hop_all<S, G, DAG, 1, WaveView16, POL>(acc, a.U, wv, g, e, i, xc);
    } else {
      hop_all<S, G, DAG, 1, SpinorView<S>, POL>(acc, a.U, in, g, e, i, xc);
    }
  }

  if constexpr (EPI == EPI_PLAIN) {
    if (active) store_spinor<S>(a.out, i, vh, acc);
  } else if constexpr (EPI == EPI_CLINV || EPI == EPI_SOLVE) {
    if (active) {
      if (a.C) {
        V r[12];
        clover_apply<G, EPI == EPI_SOLVE, POL>(r, acc, a.C, a.Cn, e, i, vh);
        store_spinor<S>(a.out, i, vh, r);
      } else {
        store_spinor<S>(a.out, i, vh, acc);
      }
    }
  } else {
    double dot = 0.0;
    if (active) {
      V x0[12], r[12];
      load_spinor<S>(x0, a.x0, i, vh);
      // the hop sum is complete; keep it from being interleaved with the
      // clover loads
      HB_SCHED_FENCE();
      if (a.C) clover_apply<G, 0, POL>(r, x0, a.C, a.Cn, e, i, vh);
      else {
#pragma unroll
        for (int k = 0; k < 12; k++) r[k] = x0[k];
      }
      const A mk2 = (A)a.mkappa2, rho = (A)a.rho;
#pragma unroll
      for (int k = 0; k < 12; k++) {
        r[k].x += mk2 * acc[k].x + rho * x0[k].x;
        r[k].y += mk2 * acc[k].y + rho * x0[k].y;
      }
      store_spinor<S>(a.out, i, vh, r);
      if constexpr (EPI == EPI_MTDOT) {
        V v[12];
        load_spinor<S>(v, a.dotv, i, vh);
#pragma unroll
        for (int k = 0; k < 12; k++) dot += (double)v[k].x * (double)r[k].x + (double)v[k].y * (double)r[k].y;
      }
    }
    if constexpr (EPI == EPI_MTDOT) {
      double vals[1] = {dot};
      block_partials<1>(vals, a.partials);
    }
  }
}

// The same for lattices with few sites per compute unit, where a kernel takes
// as long as the chain of one thread's eight hops: NW waves of a workgroup
// share 64 sites, each computes part of the hops, and the parts meet in LDS.
// Waves 0 and 1 apply one chiral block of the clover term each (to x0 before
// the barrier, or to the sum of the parts after it); wave 0 writes the result.
template <class S, class G, bool DAG, int EPI, int NW, int POL>
__global__ __launch_bounds__(64 * NW) void k_dslash_split(DslashArgs<S, G> a) {
  using V = typename S::V;
  using A = typename S::A;
  __shared__ V part[NW][12][64];
  __shared__ V y1s[EPI == EPI_PLAIN ? 1 : 6][64];
  if (a.skip && *a.skip) return;
  const Geom g = a.g;
  const int vh = g.vh, e = a.out_parity;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i = xcd_block(blockIdx.x, gridDim.x) * 64 + lane;
  const bool active = i < vh;
  constexpr bool kClovSum = EPI == EPI_CLINV || EPI == EPI_SOLVE, kClovX0 = EPI == EPI_MTIL || EPI == EPI_MTDOT;
  CloverFetch<G> cf;
  V acc[12], x0[12], y[6], dv[12];
#pragma unroll
  for (int k = 0; k < 12; k++) acc[k] = cmk<V>((A)0, (A)0);
  if (active) {
    int xc[4];
    site_coords(g, e, i, xc[0], xc[1], xc[2], xc[3]);
    const SpinorView<S> in(a.in, vh);
#define HB_PART(W) case W: if constexpr (W < NW) hop_part<S, G, DAG, NW, W % NW, POL>(acc, a.U, in, g, e, i, xc); break;
    switch (w) {
      HB_PART(0) HB_PART(1) HB_PART(2) HB_PART(3)
    }
#undef HB_PART
    if constexpr (kClovX0) {
      if (w < 2) load_spinor<S>(x0, a.x0, i, vh);
      if (w < 2 && a.C) {
        cf.template load<POL>(a.C, e, w, i, vh);
        V xp[6];
#pragma unroll
        for (int m = 0; m < 6; m++) xp[m] = w == 0 ? cadd(x0[m], x0[m + 6]) : csub(x0[m], x0[m + 6]);
        cf.template apply<0>(y, xp);
        if (w == 1) {
#pragma unroll
          for (int m = 0; m < 6; m++) y1s[m][lane] = y[m];
        }
      }
    }
    if (EPI == EPI_MTDOT && w == 0) load_spinor<S>(dv, a.dotv, i, vh);
#pragma unroll
    for (int k = 0; k < 12; k++) part[w][k][lane] = acc[k];
  }
  __syncthreads();
  if (w < (kClovSum ? 2 : 1) && active) {
#pragma unroll
    for (int k = 0; k < 12; k++) acc[k] = part[0][k][lane];
#pragma unroll
    for (int q = 1; q < NW; q++) {
#pragma unroll
      for (int k = 0; k < 12; k++) acc[k] = cadd(acc[k], part[q][k][lane]);
      HB_SCHED_FENCE();  // one part's reads in flight at a time (registers)
    }
    if (kClovSum && a.C) {
      cf.template load<POL>(a.C, e, w, i, vh);
      V xp[6];
#pragma unroll
      for (int m = 0; m < 6; m++) xp[m] = w == 0 ? cadd(acc[m], acc[m + 6]) : csub(acc[m], acc[m + 6]);
      cf.template apply<EPI == EPI_SOLVE>(y, xp);
      if (w == 1) {
#pragma unroll
        for (int m = 0; m < 6; m++) y1s[m][lane] = y[m];
      }
    }
  }
  if (kClovSum && a.C) __syncthreads();
  if (w > 0) return;
  double dot = 0.0;
  if (active) {
    V r[12];
    if (EPI != EPI_PLAIN && a.C) {
#pragma unroll
      for (int m = 0; m < 6; m++) {
        const V z = y1s[m][lane];
        r[m] = cadd(y[m], z);
        r[m + 6] = csub(y[m], z);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 12; k++) r[k] = kClovX0 ? x0[k] : acc[k];
    }
    if constexpr (kClovX0) {
      const A mk2 = (A)a.mkappa2, rho = (A)a.rho;
#pragma unroll
      for (int k = 0; k < 12; k++) {
        r[k].x += mk2 * acc[k].x + rho * x0[k].x;
        r[k].y += mk2 * acc[k].y + rho * x0[k].y;
      }
    }
    store_spinor<S, false>(a.out, i, vh, r);
    if constexpr (EPI == EPI_MTDOT) {
#pragma unroll
      for (int k = 0; k < 12; k++) dot += (double)dv[k].x * (double)r[k].x + (double)dv[k].y * (double)r[k].y;
    }
  }
  if constexpr (EPI == EPI_MTDOT) {
    dot = wave_sum(dot);
    if (lane == 0) a.partials[blockIdx.x] = dot;
  }
}

template <class S, class G, int NW, int POL>
static void launch_split(const DslashArgs<S, G> &a, bool dag, int epi, hipStream_t st) {
  dim3 grid(dslash_grid<S, G>(a.g.vh)), block(64 * NW);
#define HB_DS(D, E) hipLaunchKernelGGL((k_dslash_split<S, G, D, E, NW, POL>), grid, block, 0, st, a)
  if (!dag) {
    switch (epi) {
      case EPI_PLAIN:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(false, EPI_PLAIN);
        break;
      case EPI_CLINV: HB_DS(false, EPI_CLINV); break;
      case EPI_MTIL: HB_DS(false, EPI_MTIL); break;
      case EPI_SOLVE:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(false, EPI_SOLVE);
        break;
      default: HB_DS(false, EPI_MTDOT); break;
    }
  } else {
    switch (epi) {
      case EPI_PLAIN:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(true, EPI_PLAIN);
        break;
      case EPI_CLINV: HB_DS(true, EPI_CLINV); break;
      case EPI_MTIL: HB_DS(true, EPI_MTIL); break;
      case EPI_SOLVE:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(true, EPI_SOLVE);
        break;
      default: HB_DS(true, EPI_MTDOT); break;
    }
  }
#undef HB_DS
}

template <class S, class G, int POL>
static void launch_pol(const DslashArgs<S, G> &a, bool dag, int epi, hipStream_t st) {
  dim3 grid(dslash_grid<S, G>(a.g.vh)), block(dslash_tile<S, G>(a.g.vh));
#define HB_DS(D, E) hipLaunchKernelGGL((k_dslash<S, G, D, E, POL>), grid, block, 0, st, a)
  if (!dag) {
    switch (epi) {
      case EPI_PLAIN:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(false, EPI_PLAIN);
        break;
      case EPI_CLINV: HB_DS(false, EPI_CLINV); break;
      case EPI_MTIL: HB_DS(false, EPI_MTIL); break;
      case EPI_SOLVE:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(false, EPI_SOLVE);
        break;
      default: HB_DS(false, EPI_MTDOT); break;
    }
  } else {
    switch (epi) {
      case EPI_PLAIN:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(true, EPI_PLAIN);
        break;
      case EPI_CLINV: HB_DS(true, EPI_CLINV); break;
      case EPI_MTIL: HB_DS(true, EPI_MTIL); break;
      case EPI_SOLVE:
        if constexpr (std::is_same<G, SF64>::value) HB_DS(true, EPI_SOLVE);
        break;
      default: HB_DS(true, EPI_MTDOT); break;
    }
  }
#undef HB_DS
}

template <class S, class G>
int launch_dslash(const DslashArgs<S, G> &a, bool dag, int epi, hipStream_t st) {
  HB_CHECK((epi != EPI_PLAIN && epi != EPI_SOLVE) || (std::is_same<G, SF64>::value), HB_E_ARG,
           "launch_dslash: epilogue %d is built for FP64 links of 18 reals", epi);
  const int vh = a.g.vh, nw = split_waves<S, G>(vh);
  const bool stream = operator_policy<S, G>(vh, 1, a.C != nullptr) == kNT;
  // policies that the lines never combine with a form are not built
  constexpr int two = two_wave_sites<S, G>();
  constexpr int least = kept_sites<S, G>(true), most = kept_sites<S, G>(false);
  static_assert(least >= kFourWaveSites && most >= least, "four waves share a site where the operator is kept");
  if (nw == 4) {
    launch_split<S, G, 4, 0>(a, dag, epi, st);
  } else if (nw == 2) {
    if constexpr (least < two) {
      if (stream) launch_split<S, G, 2, kNT>(a, dag, epi, st);
      else launch_split<S, G, 2, 0>(a, dag, epi, st);
    } else {
      launch_split<S, G, 2, 0>(a, dag, epi, st);
    }
  } else {
    if constexpr (most > two) {
      if (stream) launch_pol<S, G, kNT>(a, dag, epi, st);
      else launch_pol<S, G, 0>(a, dag, epi, st);
    } else {
      launch_pol<S, G, kNT>(a, dag, epi, st);
    }
  }
  HB_HIP(hipGetLastError());
  return HB_OK;
}

template int launch_dslash<SF64, SF64>(const DslashArgs<SF64, SF64> &, bool, int, hipStream_t);
// FP64 spinors with two-row FP64 links (the FP64 CG iteration)
template int launch_dslash<SF64, SF64R>(const DslashArgs<SF64, SF64R> &, bool, int, hipStream_t);
template int launch_dslash<SF32, SF32>(const DslashArgs<SF32, SF32> &, bool, int, hipStream_t);
template int launch_dslash<SF16, SF16>(const DslashArgs<SF16, SF16> &, bool, int, hipStream_t);
// FP32 spinors with FP16 links and clover
template int launch_dslash<SF32, SF16>(const DslashArgs<SF32, SF16> &, bool, int, hipStream_t);

}  // namespace hb
