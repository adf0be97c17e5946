// Hop kernel for lattices too small to fill the device: the eight hop terms
// of a site are computed by eight wavefronts.
//
// hop_kernel gives a work-item all eight terms of its site, one load - product
// chain after the other; with one wavefront per SIMD or fewer nothing hides
// the eight load latencies. Here a work-group takes 64 sites: wavefront d < 8
// computes term d of all of them (backward, forward per dimension) and leaves
// its half spinor in LDS, so the loads of all terms are in flight at once; the
// wavefronts after them load chi and the clover block meanwhile, add the terms
// in hop_kernel's order behind one barrier, apply the epilogue and store. Every
// expression is hop_kernel's, so the results are the same bit for bit.
#pragma once

#include "hop_impl.hpp"

namespace qphix_amd {

constexpr int kSplitSites = 64;
// wavefronts of the epilogue: one per chiral block, or one per spin for the
// full blocks, whose registers (72 or 144) would cost half the work-groups
constexpr int split_epi(int kind) { return kind == KD_FULL ? 4 : 2; }
constexpr int split_threads(int kind) { return 64 * (8 + split_epi(kind)); }
// the results meet in LDS before the store: the half precisions scale a site's
// values by the largest of them, and a spin of FP32 is a word and a half
constexpr bool split_gather(int p, int kind) { return p == P16 || p == PB16 || (p == P32 && kind == KD_FULL); }

// Largest number of sites (times right-hand sides) that take this form by
// rule; from 2^17 sites on, where the hops are tuned, it is a candidate of the
// tuner instead. The lines lie where the forms meet: in FP64 and the half
// precisions, and for full blocks, below a wavefront per SIMD of hop_kernel (65536
// sites), whose wider loads per wavefront then begin to pay; FP32 keeps its
// lead to the tuner's range. Measured in us, hop_kernel / this, with the fields
// in the caches and (in brackets) after 1.2 GB of other traffic, the launch's 3 us
// included there. A^-1 D psi, FP64: 2048 sites 10.4 / 5.1 (13.7 / 7.7), 13824
// 16.8 / 5.7 (20.0 / 9.4), 32768 19.2 / 14.1 (22.0 / 16.8), 49152 20.9 / 19.9
// (24.0 / 22.4), 65536 23.8 / 24.8; FP32: 2048 7.6 / 4.4 (10.6 / 7.0), 32768
// 12.4 / 5.6 (15.4 / 9.4), 65536 14.1 / 11.8 (17.2 / 14.6), 115200 21.0 / 18.9
// (24.1 / 21.8), 331776 51.8 / 48.5; FP16: 2048 7.2 / 4.8 (10.1 / 7.4), 32768
// 8.6 / 6.0 (12.0 / 8.8), 40960 9.3 / 8.4 (12.5 / 11.4), 65536 9.7 / 11.3. The
// Wilson hop gains least: FP64 49152 17.1 / 16.5 and, on 16x16x24x16, 17.4 / 17.2
// (19.8 / 19.8, 20.2 / 21.0), FP16 36960 7.3 / 7.6 (10.8 / 10.4). Full blocks:
// FP64 49152 24.7 / 23.7 (27.8 / 26.5), FP32 49152 14.6 / 12.6 (17.9 / 15.3), 65536
// 15.6 / 15.5, FP16 32768 9.9 / 6.0 (13.2 / 9.4), 40960 10.5 / 8.3 (13.6 / 12.0).
constexpr long split_sites(int p, int kind) {
  return p == P64 ? 49152 : p == P32 ? (kind == KD_FULL ? 49152 : (1l << 17) - 1) : 45056;
}
inline bool use_split(int p, int kind, const HopArgs &a, int nr) {
  if (kind == KD_DIR || a.bz != 0 || a.split < 0) return false;
  return a.split > 0 || (long)a.vh * nr <= split_sites(p, kind);
}

// one term: lds[k * 64 + lane] gets the 12 reals of coef U h
template <int P, bool C12, int ISIGN, int MU, bool FWD>
__device__ inline void split_term(const HopArgs &a, const void *psi_p, unsigned s, unsigned sn,
                                  typename PT<P>::calc coef, typename PT<P>::calc *lds) {
  typedef typename PT<P>::calc T;
  typedef GaugeLayout<P, C12> GL;
  constexpr int S = FWD ? -ISIGN : ISIGN;
  // the words that hold the link
  constexpr int pw = PT<P>::per_word;
  constexpr int first = (2 * MU + (FWD ? 1 : 0)) * GL::link_reals;
  constexpr int w0 = first / pw, nwl = (first + GL::link_reals + pw - 1) / pw - w0;
  const bool tbc = (a.tbc_mask >> MU) & 1;
  T tr = tbc ? (T)a.tbc_r[MU] : (T)1, ti = tbc ? (T)a.tbc_i[MU] : (T)0;
  T sp[kSpinorReals], lv[nwl * pw];
  load_spinor<P, false, !PT<P>::scaled>(psi_p, a.vs, sn, sp);
  load_range<P, GL::nw, w0, nwl, false, !PT<P>::scaled>(a.u, a.vs, s, lv);
  cx<T> psi[4][3], U[3][3], h[2][3], uh[2][3];
  to_spinor(sp, psi);
  if constexpr (PT<P>::scaled) {
    const T su = site_scale<P>(a.u, a.vs, s, GL::nw);
    const T f = su * site_scale<P>(psi_p, a.vs, sn, words_of<P>(kSpinorReals));
    make_link<C12>(lv + (first - w0 * pw), U, su);
    tr = tr * f;
    ti = ti * f;
  } else {
    make_link<C12>(lv + (first - w0 * pw), U);
  }
  project<MU, S>(psi, h);
  link_times_half<FWD, fma_of<P>()>(U, h, tr, ti, uh);
#pragma unroll
  for (int r = 0; r < 2; r++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const cx<T> v = scale(coef, uh[r][c]);
      lds[(6 * r + 2 * c) * kSplitSites] = v.r;
      lds[(6 * r + 2 * c + 1) * kSplitSites] = v.i;
    }
}

// acc[s - S0] += the reconstruction of one term on spins S0 .. S0 + NS - 1
template <int MU, bool FWD, int ISIGN, int S0, int NS, typename T>
__device__ inline void split_add(const T *lds, cx<T> (&acc)[NS][3]) {
  constexpr int S = FWD ? -ISIGN : ISIGN;
#pragma unroll
  for (int q = 0; q < NS; q++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const int row = S0 + q;
      const int r = row < 2 ? row : gcol(MU, row);
      const cx<T> v = mk(lds[(6 * r + 2 * c) * kSplitSites], lds[(6 * r + 2 * c + 1) * kSplitSites]);
      if (row < 2) acc[q][c] = acc[q][c] + v;
      else if (row == 2) acc[q][c] = acc[q][c] + mulph<S * gpr(MU, 2), S * gpi(MU, 2)>(v);
      else acc[q][c] = acc[q][c] + mulph<S * gpr(MU, 3), S * gpi(MU, 3)>(v);
    }
}
template <int ISIGN, int S0, int NS, typename T>
__device__ inline void split_sum(const T *lds, cx<T> (&acc)[NS][3]) {
  constexpr int D = 12 * kSplitSites;
  split_add<0, false, ISIGN, S0, NS>(lds, acc);
  split_add<0, true, ISIGN, S0, NS>(lds + D, acc);
  split_add<1, false, ISIGN, S0, NS>(lds + 2 * D, acc);
  split_add<1, true, ISIGN, S0, NS>(lds + 3 * D, acc);
  split_add<2, false, ISIGN, S0, NS>(lds + 4 * D, acc);
  split_add<2, true, ISIGN, S0, NS>(lds + 5 * D, acc);
  split_add<3, false, ISIGN, S0, NS>(lds + 6 * D, acc);
  split_add<3, true, ISIGN, S0, NS>(lds + 7 * D, acc);
}

// reals [R0, R0 + N) of a field: loads the words that hold them
template <int P, int NWT, int R0, int N, bool SCALED>
__device__ inline void load_reals(const void *base, size_t vs, long s, typename PT<P>::calc (&o)[N]) {
  constexpr int pw = PT<P>::per_word;
  constexpr int w0 = R0 / pw, nw = (R0 + N + pw - 1) / pw - w0;
  typename PT<P>::calc v[nw * pw];
  load_range<P, NWT, w0, nw, false, SCALED>(base, vs, s, v);
#pragma unroll
  for (int k = 0; k < N; k++) o[k] = v[R0 - w0 * pw + k];
}

// Epilogue of spins 2 B, 2 B + 1 (chiral block B), as hop_init_r and
// hop_finish_r; H >= 0: only spin 2 B + H of the result (KD_FULL)
template <int P, int ISIGN, int KIND, int B, int H>
__device__ inline void split_epilogue(const HopArgs &a, const typename PT<P>::calc *lds, typename PT<P>::calc *res,
                                      const void *chi_p, void *out_p, unsigned s, bool live) {
  typedef typename PT<P>::calc T;
  constexpr bool raw = PT<P>::scaled;
  constexpr bool has_chi = KIND == KA_WILSON || KIND == KA_CLOVER || KIND == KA_TM;
  constexpr int nws = words_of<P>(kSpinorReals), nwc = words_of<P>(kCloverReals), nwf = words_of<P>(kFullCloverReals);
  constexpr int rows = H < 0 ? 6 : 3, row0 = H < 0 ? 0 : 3 * H;
  cx<T> acc[2][3], ch[2][3];
  T m[KIND == KD_CLOVER || KIND == KA_CLOVER ? 36 : 1], f[KIND == KD_FULL ? 12 * rows : 1];
  T sc = (T)1;
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int c = 0; c < 3; c++) acc[q][c] = mk((T)0, (T)0);
  if (live) {
    if constexpr (KIND == KD_CLOVER || KIND == KA_CLOVER) {
      load_reals<P, nwc, 36 * B, 36, !raw>(a.clov, a.vs, s, m);
      if constexpr (raw) sc = site_scale<P>(a.clov, a.vs, s, nwc);
    }
    if constexpr (KIND == KD_FULL) {
      load_reals<P, nwf, 72 * B + 12 * row0, 12 * rows, !raw>(a.clov, a.vs, s, f);
      if constexpr (raw) sc = site_scale<P>(a.clov, a.vs, s, nwf);
    }
    if constexpr (has_chi) {
      T cv[12];
      load_reals<P, nws, 12 * B, 12, true>(chi_p, a.vs, s, cv);
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int c = 0; c < 3; c++) ch[q][c] = mk(cv[6 * q + 2 * c], cv[6 * q + 2 * c + 1]);
    }
  }
  auto ig5 = [&](T g, const cx<T> (&in)[2][3], cx<T> (&out)[2][3]) {
    const T gg = B == 0 ? g : -g;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) out[q][c] = out[q][c] + mk(-gg * in[q][c].i, gg * in[q][c].r);
  };
  if constexpr (KIND == KA_WILSON) {
    const T al = (T)a.alpha;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) acc[q][c] = scale(al, ch[q][c]);
  } else if constexpr (KIND == KA_CLOVER) {
    cx<T> v[6], w[6];
#pragma unroll
    for (int i = 0; i < 6; i++) v[i] = ch[i / 3][i % 3];
    herm6<false>(m, v, w);
#pragma unroll
    for (int i = 0; i < 6; i++) acc[i / 3][i % 3] = raw ? scale(sc, w[i]) : w[i];
    ig5((T)(ISIGN * a.rho), ch, acc);
  } else if constexpr (KIND == KA_TM) {
    const T al = (T)a.alpha;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) acc[q][c] = ch[q][c];
    ig5((T)(ISIGN * a.mu), ch, acc);
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) acc[q][c] = scale(al, acc[q][c]);
  }
  __syncthreads();  // the eight terms are in LDS
  if (!live) return;
  split_sum<ISIGN, 2 * B, 2>(lds, acc);
  T o[2 * rows];
  if constexpr (KIND == KD_CLOVER || KIND == KD_FULL) {
    cx<T> v[6];
#pragma unroll
    for (int i = 0; i < 6; i++) v[i] = acc[i / 3][i % 3];
    if constexpr (KIND == KD_CLOVER) {
      cx<T> w[6];
      herm6<fma_of<P>()>(m, v, w);
#pragma unroll
      for (int i = 0; i < 6; i++) {
        const cx<T> x = raw ? scale(sc, w[i]) : w[i];
        o[2 * i] = x.r;
        o[2 * i + 1] = x.i;
      }
    } else {
      cx<T> w[rows];
      full6_rows<fma_of<P>()>(f, v, w);
#pragma unroll
      for (int i = 0; i < rows; i++) {
        const cx<T> x = raw ? scale(sc, w[i]) : w[i];
        o[2 * i] = x.r;
        o[2 * i + 1] = x.i;
      }
    }
  } else {
    cx<T> x[2][3];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) x[q][c] = acc[q][c];
    if constexpr (KIND == KD_TM) {
      ig5((T)(-ISIGN * a.mu), acc, x);
      const T mi = (T)a.muinv;
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int c = 0; c < 3; c++) x[q][c] = scale(mi, x[q][c]);
    }
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        o[6 * q + 2 * c] = x[q][c].r;
        o[6 * q + 2 * c + 1] = x[q][c].i;
      }
  }
  if constexpr (split_gather(P, KIND)) {
#pragma unroll
    for (int k = 0; k < 2 * rows; k++) res[(12 * B + 2 * row0 + k) * kSplitSites] = o[k];
  } else {
    constexpr int pw = PT<P>::per_word, w0 = (12 * B + 2 * row0) / pw;
#pragma unroll
    for (int w = 0; w < 2 * rows / pw; w++) Word<P>::template store<true>(out_p, widx(s, w0 + w, nws), o + w * pw);
  }
}

// three work-groups of ten wavefronts to a CU (64 registers) where a spill-free
// allocation gives them
constexpr int split_min_waves(int p, int kind) {
  return (p == P16 || p == PB16) && kind != KD_FULL && kind != KD_CLOVER ? 8 : 1;
}

template <int P, bool C12, int ISIGN, int KIND>
__global__ void __launch_bounds__(split_threads(KIND), split_min_waves(P, KIND)) hop_split_kernel(const HopArgs a) {
  if (a.skip && *a.skip) return;
  typedef typename PT<P>::calc T;
  __shared__ T terms[8 * 12 * kSplitSites];
  __shared__ T result[split_gather(P, KIND) ? 24 * kSplitSites : 1];
  int lb = xcd_block();
  const void *psi_p = a.psi, *chi_p = a.chi;
  void *out_p = a.out;
  if (a.nrhs > 1) {
    const int r = lb % a.nrhs;
    lb /= a.nrhs;
    const HopArgs *ka = (const HopArgs *)__builtin_amdgcn_kernarg_segment_ptr();  // as in hop_kernel
    psi_p = ka->psis[r];
    out_p = ka->outs[r];
    chi_p = ka->chis[r];
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const unsigned s = (unsigned)lb * kSplitSites + lane;
  const bool live = s < (unsigned)a.vh;
  T *res = result + (split_gather(P, KIND) ? lane : 0);
  if (wave < 8) {
    if (live) {
      T *lds = terms + wave * 12 * kSplitSites + lane;
      const SiteNbrs n = site_nbrs(a, s);
      const T cs = (T)a.cs;
      switch (wave) {
        case 0: split_term<P, C12, ISIGN, 0, false>(a, psi_p, s, n.xb, cs, lds); break;
        case 1: split_term<P, C12, ISIGN, 0, true>(a, psi_p, s, n.xf, cs, lds); break;
        case 2: split_term<P, C12, ISIGN, 1, false>(a, psi_p, s, n.yb, cs, lds); break;
        case 3: split_term<P, C12, ISIGN, 1, true>(a, psi_p, s, n.yf, cs, lds); break;
        case 4: split_term<P, C12, ISIGN, 2, false>(a, psi_p, s, n.zb, cs, lds); break;
        case 5: split_term<P, C12, ISIGN, 2, true>(a, psi_p, s, n.zf, cs, lds); break;
        case 6: split_term<P, C12, ISIGN, 3, false>(a, psi_p, s, n.tb, (T)(n.t_lo ? a.ctb : a.ct), lds); break;
        default: split_term<P, C12, ISIGN, 3, true>(a, psi_p, s, n.tf, (T)(n.t_hi ? a.ctf : a.ct), lds); break;
      }
    }
    __syncthreads();
  } else if constexpr (split_epi(KIND) == 2) {
    if (wave == 8) split_epilogue<P, ISIGN, KIND, 0, -1>(a, terms + lane, res, chi_p, out_p, s, live);
    else split_epilogue<P, ISIGN, KIND, 1, -1>(a, terms + lane, res, chi_p, out_p, s, live);
  } else {
    if (wave == 8) split_epilogue<P, ISIGN, KIND, 0, 0>(a, terms + lane, res, chi_p, out_p, s, live);
    else if (wave == 9) split_epilogue<P, ISIGN, KIND, 0, 1>(a, terms + lane, res, chi_p, out_p, s, live);
    else if (wave == 10) split_epilogue<P, ISIGN, KIND, 1, 0>(a, terms + lane, res, chi_p, out_p, s, live);
    else split_epilogue<P, ISIGN, KIND, 1, 1>(a, terms + lane, res, chi_p, out_p, s, live);
  }
  if constexpr (split_gather(P, KIND)) {
    __syncthreads();
    if (wave < words_of<P>(kSpinorReals) && live) {  // a word per wavefront, as store_all
      constexpr int pw = PT<P>::per_word, nws = words_of<P>(kSpinorReals);
      T t[pw];
      if constexpr (PT<P>::scaled) {
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < kSpinorReals; k++) m = fmaxf(m, fabsf(res[k * kSplitSites]));
        const float inv = m > 0.f ? 1.0f / m : 0.f;
#pragma unroll
        for (int k = 0; k < pw; k++) t[k] = res[(wave * pw + k) * kSplitSites] * inv;
        if (wave == 0) reinterpret_cast<float *>(reinterpret_cast<char *>(out_p) + (size_t)nws * a.vs * 16)[s] = m;
      } else {
#pragma unroll
        for (int k = 0; k < pw; k++) t[k] = res[(wave * pw + k) * kSplitSites];
      }
      Word<P>::template store<true>(out_p, widx(s, wave, nws), t);
    }
  }
}

}  // namespace qphix_amd
