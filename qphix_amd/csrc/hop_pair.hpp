// Hops of a non-degenerate flavour doublet: both flavours in one launch, with
// the flavour-mixing epilogue.
//
// The doublet operators are two Wilson hops, a 2 x 2 flavour matrix of site
// terms, two A chi - D psi hops and a flavour-crossed chi (tm_dslash_body.h:344-367,
// tm_clov_dslash_body.h:1262-1367, ndtm_reuse_operator*.h). One launch per half: a
// work-group takes 128 sites, its first two wavefronts the up flavour, the
// others the down one, so the links (and the flavour-independent clover
// blocks) are read from memory once for both, the hop results meet in LDS
// instead of going to memory and back, and chi of the other flavour joins the
// accumulator instead of taking a pass of its own. Bound: links and site
// terms. Measured per TM-clover doublet operator, separate passes / this, us:
// 8^4 FP64 57 / 26, 16^3x32 FP64 155 / 104, FP32 91 / 46, FP16 67 / 33,
// 32^3x48 FP64 1676 / 1158, FP32 750 / 510, FP16 450 / 318; the Wilson doublet
// gains alike (109 / 65 at 16^3x32 FP64).
// Where nothing is rounded to half storage in between, the results are the
// separate passes' bit for bit.
#pragma once

#include "hop_impl.hpp"

namespace qphix_amd {

// out_f = F_f D psi_f + C D psi_f'; out_f = (a0 +- i a1 g5) D psi_f + e D psi_f';
// A chi_f +- i rho g5 chi_f - b D psi_f - eps chi_f'; the same with alpha (1 +- i mu g5)
enum PairKind { PD_CLOVER = 0, PD_TM, PA_CLOVER, PA_TM };

struct PairArgs {
  HopArgs a;         // first: read in place from the kernel-argument segment (psis, outs, chis of both flavours)
  const void *f[2];  // PD_CLOVER: full blocks of each flavour (a.clov: the off-diagonal ones)
  double t0, t1;     // PD_TM: a0 and a1 (+ for up, - for down)
  double eps;        // PD_TM: e; PA: eps
};

constexpr int kPairSites = 128;

template <int P, bool C12, int ISIGN, int KIND>
__global__ void __launch_bounds__(2 * kPairSites) hop_pair_kernel(const PairArgs pa) {
  if (pa.a.skip && *pa.a.skip) return;
  typedef typename PT<P>::calc T;
  constexpr bool mix = KIND == PD_CLOVER || KIND == PD_TM;
  constexpr int HK = KIND == PA_CLOVER ? (int)KA_CLOVER : KIND == PA_TM ? (int)KA_TM : (int)KD_WILSON;
  __shared__ T lds[mix ? kSpinorReals * 2 * kPairSites : 1];
  const PairArgs *ka = (const PairArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  const int fl = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kPairSites);
  const unsigned k = (unsigned)xcd_block() * kPairSites + (threadIdx.x & (kPairSites - 1));
  const HopArgs &a = pa.a;
  const bool live = k < (unsigned)a.vh;
  const bool wave_full = __ballot(live) == ~0ull;
  const void *const psi[1] = {ka->a.psis[fl]};
  const void *const chi[1] = {ka->a.chis[fl]};
  void *const out[1] = {ka->a.outs[fl]};
  cx<T> acc[1][4][3];
  unsigned s = 0;
  if (live) {
    const SiteNbrs n = site_nbrs(a, k);
    s = n.s;
    const T cs = (T)a.cs;
    const T ctb = (T)(n.t_lo ? a.ctb : a.ct), ctf = (T)(n.t_hi ? a.ctf : a.ct);
    const double sgn = fl ? -1.0 : 1.0;  // the twisted mass of the down flavour
    hop_init_r<P, ISIGN, HK, 1, false>(a, s, chi, acc, sgn);
    if (hop_shfl(P, HK) && wave_full) {
      T ov[kSpinorReals];
      cx<T> own[4][3];
      load_spinor<P>(psi[0], a.vs, s, ov);
      to_spinor(ov, own);
      const unsigned s0 = __shfl(s, 0, 64);
      const bool contig = __shfl(s, 63, 64) == s0 + 63u;
      hop_dim_shfl<P, C12, ISIGN, 0, false>(a, psi[0], own, s, n.xb, n.xf, s0, contig, cs, acc[0]);
      hop_dim_shfl<P, C12, ISIGN, 1, false>(a, psi[0], own, s, n.yb, n.yf, s0, contig, cs, acc[0]);
    } else {
      hop_dim<P, C12, ISIGN, 0, false>(a, psi[0], s, n.xb, n.xf, cs, cs, acc[0]);
      hop_dim<P, C12, ISIGN, 1, false>(a, psi[0], s, n.yb, n.yf, cs, cs, acc[0]);
    }
    hop_dim<P, C12, ISIGN, 2, false>(a, psi[0], s, n.zb, n.zf, cs, cs, acc[0]);
    hop_dim<P, C12, ISIGN, 3, false>(a, psi[0], s, n.tb, n.tf, ctb, ctf, acc[0]);
  }
  T ov[kSpinorReals];
  if constexpr (mix) {
    // both flavours of a site: lanes t and t ^ 128
    if (live) {
      from_spinor(acc[0], ov);
#pragma unroll
      for (int e = 0; e < kSpinorReals; e++) lds[e * 2 * kPairSites + threadIdx.x] = ov[e];
    }
    __syncthreads();
    if (!live) return;
    cx<T> other[1][4][3], o[1][4][3];
#pragma unroll
    for (int e = 0; e < kSpinorReals; e++) ov[e] = lds[e * 2 * kPairSites + (threadIdx.x ^ kPairSites)];
    to_spinor(ov, other[0]);
    if constexpr (KIND == PD_CLOVER) {
      cx<T> c[1][4][3];
      full_block_apply_r<P, 0, 1>(ka->f[fl], a.vs, s, acc, o);
      full_block_apply_r<P, 1, 1>(ka->f[fl], a.vs, s, acc, o);
      clover_block_apply_r<P, 0, 1, fma_of<P>(), false>(a.clov, a.vs, s, other, c);
      clover_block_apply_r<P, 1, 1, fma_of<P>(), false>(a.clov, a.vs, s, other, c);
#pragma unroll
      for (int sp = 0; sp < 4; sp++)
#pragma unroll
        for (int cc = 0; cc < 3; cc++) o[0][sp][cc] = o[0][sp][cc] + c[0][sp][cc];
    } else {
      const T a0 = (T)pa.t0, a1 = (T)(fl ? -pa.t1 : pa.t1), e = (T)pa.eps;
#pragma unroll
      for (int sp = 0; sp < 4; sp++) {
        const T g = sp < 2 ? a1 : -a1;
#pragma unroll
        for (int cc = 0; cc < 3; cc++) {
          const cx<T> u = acc[0][sp][cc], d = other[0][sp][cc];
          o[0][sp][cc] = mk(a0 * u.r - g * u.i + e * d.r, a0 * u.i + g * u.r + e * d.i);
        }
      }
    }
    from_spinor(o[0], ov);
  } else {
    if (!live) return;
    // half storage: the stored values pinned and scaled here (as the hops read
    // theirs); read scaled, the load took the kernel from 129 registers to 244
    from_spinor(acc[0], ov);
    const T e = (T)-pa.eps;
    T ch[kSpinorReals];
    load_spinor<P, false, false>(ka->a.chis[1 - fl], a.vs, s, ch);
    const T sc = PT<P>::scaled ? site_scale<P>(ka->a.chis[1 - fl], a.vs, s, words_of<P>(kSpinorReals)) : (T)1;
#pragma unroll
    for (int i = 0; i < kSpinorReals; i++) ov[i] = e * (PT<P>::scaled ? sc * ch[i] : ch[i]) + ov[i];
  }
  store_spinor<P, true>(out[0], a.vs, s, ov);
}

template <int P, bool C12, int ISIGN>
static hipError_t launch_pair3(int kind, const PairArgs &pa, hipStream_t st) {
  const unsigned grid = (unsigned)((pa.a.vh + kPairSites - 1) / kPairSites);
  switch (kind) {
#define PK(K) \
  case K: hop_pair_kernel<P, C12, ISIGN, K><<<grid, 2 * kPairSites, 0, st>>>(pa); break;
    PK(PD_CLOVER) PK(PD_TM) PK(PA_CLOVER) PK(PA_TM)
#undef PK
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int P> hipError_t launch_hop_pair_prec(int kind, bool c12, int isign, const PairArgs &pa, hipStream_t st) {
  if (c12) return isign > 0 ? launch_pair3<P, true, 1>(kind, pa, st) : launch_pair3<P, true, -1>(kind, pa, st);
  if constexpr (!PT<P>::scaled)
    return isign > 0 ? launch_pair3<P, false, 1>(kind, pa, st) : launch_pair3<P, false, -1>(kind, pa, st);
  return hipErrorInvalidValue;
}

}  // namespace qphix_amd
