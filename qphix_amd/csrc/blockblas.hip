// Block (multi-RHS) BLAS for block Krylov solvers: the Gram matrix of two sets
// of spinor fields and the combination of one set by a small dense matrix.
//
// Both are contractions over sources or over sites with n x n results, so they
// run on the matrix cores in the storage precision (v_mfma_f32_16x16x4f32,
// v_mfma_f64_16x16x4f64), a complex product as four real ones. The operands
// go from the fields to the registers in the layout the instruction wants:
// sixteen lanes of a wavefront read sixteen consecutive sites of one 16-byte
// word (256 contiguous bytes) of a field, so there is no LDS staging and no
// barrier. Operand layouts (checked on the device by a probe): lane l gives
// A[row l % 16][k = l / 16] and B[k = l / 16][column l % 16], and holds rows
// 4 (l / 16) + r of column l % 16 of the FP32 result, rows l / 16 + 4 r of the
// FP64 one. Partial Gram matrices are summed in FP64 in a fixed order, so
// results do not depend on timing.
#include "blockblas.hpp"

namespace qphix_amd {

constexpr int kBlockThreads = 256;
constexpr int kBlockWaves = kBlockThreads / 64;

typedef double d4_t __attribute__((ext_vector_type(4)));
template <int P> struct Mfma;
template <> struct Mfma<P32> {
  typedef f4_t acc;
  __device__ static inline acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // row of the result's element r in lane group lg = lane / 16
  __device__ static constexpr int row(int lg, int r) { return 4 * lg + r; }
};
template <> struct Mfma<P64> {
  typedef d4_t acc;
  __device__ static inline acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static constexpr int row(int lg, int r) { return lg + 4 * r; }
};
template <typename A> __device__ inline A zero_acc() { return A{0, 0, 0, 0}; }

// A unit is S consecutive sites of one word, in the fields' memory order, so
// the wavefronts in flight read each field as one stream. First site of unit
// u; nsites is the end of the last whole 64-site group (the padding sites up to
// it are zero and stay so), units of layout-block padding past it are skipped.
template <int S> __device__ inline long unit_site(int u, int words) {
  constexpr int per = (int)(kSiteBlock / S);
  return (long)(u / per / words) * kSiteBlock + (long)(u % per) * S;
}

// ---------------------------------------------------------------------------
// Gram matrix G_ij = sum conj(a_i) b_j, tiles of 16 x 16 pairs
//
// Rows and columns are fields, the contraction runs over sites: a step takes
// 16 sites of one word of all fields (lane l: field l % 16, sites 4 q + l / 16,
// 64 contiguous bytes of a field per four lanes) and three accumulators per
// tile, Re Re + Im Im, Re Im and Im Re. FP32 sums are carried over 32 sites of a
// word and then added in FP64 (the vector form before it summed 64 sites in
// FP32). With both sets the same fields only the tiles on and above the diagonal are
// computed; the rest is their conjugate, exactly. Bound: the fields' reads.
// Measured at 24^3x48, FP32, 28 sources: 0.50 ms (0.28 ms for one set
// with itself) and 0.016 ms to finalize; the LDS-staged vector form took
// 1.40 ms and its one-thread-per-element finalize 0.21 ms. Error against 64
// bits 0.5 to 0.9 times that form's for 2 to 28 fields in both precisions.
// ---------------------------------------------------------------------------
constexpr int kGramTile = 16;
constexpr int kGramSites = 32;  // sites of a word between two FP64 additions

template <int P, int IT, int JT, bool SAME>
__global__ void __launch_bounds__(kBlockThreads) k_block_gram(const BlockArgs ba, long nsites, int nunits, double *partials) {
  typedef typename PT<P>::calc T;
  typedef Mfma<P> M;
  typedef typename M::acc Acc;
  constexpr int W = words_of<P>(kSpinorReals);
  constexpr int PW = PT<P>::per_word;
  constexpr int CW = PW / 2;
  constexpr int NT = kMaxRhs * kMaxRhs * 2;
  // the pointer tables are read in place from the kernel-argument segment
  // (BlockArgs is the first parameter): a run-time index into the by-value
  // parameter would copy it to private memory
  const BlockArgs *ka = (const BlockArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lc = lane & 15, lg = lane >> 4;
  // rows and columns past the sets read the last field and are not stored
  const void *pa[IT], *pb[JT];
#pragma unroll
  for (int i = 0; i < IT; i++) pa[i] = ka->a[i * kGramTile + lc < ba.na ? i * kGramTile + lc : ba.na - 1];
#pragma unroll
  for (int j = 0; j < JT; j++)
    pb[j] = SAME ? pa[j < IT ? j : 0] : ka->b[j * kGramTile + lc < ba.nb ? j * kGramTile + lc : ba.nb - 1];

  double gr[IT][JT][4], gi[IT][JT][4];
#pragma unroll
  for (int i = 0; i < IT; i++)
#pragma unroll
    for (int j = 0; j < JT; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) gr[i][j][r] = gi[i][j][r] = 0.0;

  for (int u = blockIdx.x * kBlockWaves + wave; u < nunits; u += gridDim.x * kBlockWaves) {
    if (unit_site<kGramSites>(u, W) >= nsites) continue;
    Acc rr[IT][JT], ri[IT][JT], ir[IT][JT];
#pragma unroll
    for (int i = 0; i < IT; i++)
#pragma unroll
      for (int j = 0; j < JT; j++) rr[i][j] = ri[i][j] = ir[i][j] = zero_acc<Acc>();
#pragma unroll
    for (int h = 0; h < kGramSites / 16; h++) {
      T va[IT][4][PW], vb[JT][4][PW];
      const size_t wi = (size_t)u * kGramSites + h * 16 + lg;
#pragma unroll
      for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int i = 0; i < IT; i++) Word<P>::template load<false>(pa[i], wi + 4 * q, va[i][q]);
        if constexpr (!SAME) {
#pragma unroll
          for (int j = 0; j < JT; j++) Word<P>::template load<false>(pb[j], wi + 4 * q, vb[j][q]);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int c = 0; c < CW; c++)
#pragma unroll
          for (int i = 0; i < IT; i++)
#pragma unroll
            for (int j = 0; j < JT; j++) {
              if (SAME && i > j) continue;
              const T ar = va[i][q][2 * c], ai = va[i][q][2 * c + 1];
              const T br = SAME ? va[j][q][2 * c] : vb[j][q][2 * c];
              const T bi = SAME ? va[j][q][2 * c + 1] : vb[j][q][2 * c + 1];
              rr[i][j] = M::mma(ar, br, rr[i][j]);
              ri[i][j] = M::mma(ar, bi, ri[i][j]);
              ir[i][j] = M::mma(ai, br, ir[i][j]);
              rr[i][j] = M::mma(ai, bi, rr[i][j]);
            }
    }
#pragma unroll
    for (int i = 0; i < IT; i++)
#pragma unroll
      for (int j = 0; j < JT; j++) {
        if (SAME && i > j) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          gr[i][j][r] += (double)rr[i][j][r];
          gi[i][j][r] += (double)ri[i][j][r] - (double)ir[i][j][r];
        }
      }
  }
  // the work-group's waves, in order
  __shared__ double sum[NT];
  for (int k = 0; k < kBlockWaves; k++) {
    if (wave == k) {
#pragma unroll
      for (int i = 0; i < IT; i++)
#pragma unroll
        for (int j = 0; j < JT; j++) {
          if (SAME && i > j) continue;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            double *o = sum + ((i * kGramTile + M::row(lg, r)) * kMaxRhs + j * kGramTile + lc) * 2;
            o[0] = k ? o[0] + gr[i][j][r] : gr[i][j][r];
            o[1] = k ? o[1] + gi[i][j][r] : gi[i][j][r];
          }
        }
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < NT; e += kBlockThreads) {
    const int i = e / (2 * kMaxRhs), j = (e >> 1) & (kMaxRhs - 1);
    if (i < ba.na && j < ba.nb && !(SAME && i / kGramTile > j / kGramTile)) partials[(size_t)blockIdx.x * NT + e] = sum[e];
  }
}

// out[(i * nb + j) * 2 + {re, im}] = sum over work-groups: 16 elements per
// work-group, each summed in 16 interleaved slices that are added in order
template <bool SAME>
__global__ void __launch_bounds__(256) k_block_gram_finalize(const double *partials, int nblocks, int na, int nb,
                                                             double *out) {
  __shared__ double part[16][17];
  const int el = threadIdx.x & 15, sl = threadIdx.x >> 4;
  const int e = blockIdx.x * 16 + el;
  const int ij = e >> 1, ri = e & 1;
  int i = ij / nb, j = ij - i * nb;
  double sgn = 1.0;
  if (SAME && i / kGramTile > j / kGramTile) {  // the conjugate of the tile above the diagonal
    const int t = i;
    i = j;
    j = t;
    sgn = ri ? -1.0 : 1.0;
  }
  double s = 0;
  if (e < na * nb * 2)
    for (int b = sl; b < nblocks; b += 16)
      s += partials[((size_t)b * kMaxRhs * kMaxRhs + i * kMaxRhs + j) * 2 + ri];
  part[sl][el] = s;
  __syncthreads();
  if (sl == 0 && e < na * nb * 2) {
    double t = 0;
    for (int k = 0; k < 16; k++) t += part[k][el];
    out[e] = sgn * t;
  }
}

// ---------------------------------------------------------------------------
// combination o_j = y_j + sum_i a_i m_ij
//
// Rows are outputs, columns sites, the contraction runs over the fields a_i:
// a step takes 16 sites of one word of every field, KG groups of four fields
// (lane l: field 4 g + l / 16, site l % 16), and JT tiles of 16 outputs. The
// matrix stays in registers. The four real products have a chain of their own
// each: one chain for two of them rounds at the size of their sum (1.3 times
// the error of the vector form before it; this form 0.95 times).
// A wavefront loads the words of all fields of its sites before it stores any,
// and no other touches them, so outputs may alias inputs. The addend joins
// the finished sum, rounded once: it is much larger than the sum where a
// solver adds corrections to a solution, and each step of the sum would round
// at its size. Bound: the fields'
// reads and writes (at 28 sources 67 kflop a site, 0.6 of the time these
// take, at the FP32 matrix peak). Measured at 24^3x48, FP32, 28 sources: 0.48 ms
// a combination (three in four with an addend, 83% of the stream rate); the
// LDS-staged vector form, which read LDS for every product, took 1.04 ms.
// ---------------------------------------------------------------------------
constexpr int kCombineSites = 16;

template <int P, int KG, int JT>
__global__ void __launch_bounds__(kBlockThreads) k_block_combine(const BlockArgs ba, long nsites, int nunits,
                                                                const double *mat) {
  typedef typename PT<P>::calc T;
  typedef Mfma<P> M;
  typedef typename M::acc Acc;
  constexpr int W = words_of<P>(kSpinorReals);
  constexpr int PW = PT<P>::per_word;
  constexpr int CW = PW / 2;
  const BlockArgs *ka = (const BlockArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  const int na = ba.na, nb = ba.nb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lc = lane & 15, lg = lane >> 4;
  // fields past the set read the last one and are multiplied by nothing
  const void *pa[KG];
  bool use[KG];
  T mr[KG][JT], mi[KG][JT];
#pragma unroll
  for (int g = 0; g < KG; g++) {
    const int i = 4 * g + lg;
    use[g] = i < na;
    pa[g] = ka->a[use[g] ? i : na - 1];
#pragma unroll
    for (int t = 0; t < JT; t++) {
      const int j = 16 * t + lc;
      const bool in = use[g] && j < nb;
      mr[g][t] = in ? (T)mat[(i * nb + j) * 2] : (T)0;
      mi[g][t] = in ? (T)mat[(i * nb + j) * 2 + 1] : (T)0;
    }
  }
  const void *py[JT][4];
  void *po[JT][4];
#pragma unroll
  for (int t = 0; t < JT; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int j = 16 * t + M::row(lg, r);
      po[t][r] = j < nb ? ka->o[j] : nullptr;
      py[t][r] = j < nb ? ka->y[j] : nullptr;
    }
  for (int u = blockIdx.x * kBlockWaves + wave; u < nunits; u += gridDim.x * kBlockWaves) {
    if (unit_site<kCombineSites>(u, W) >= nsites) continue;
    const size_t wi = (size_t)u * kCombineSites + lc;
    T va[KG][PW];
    Acc rr[JT][CW], ii[JT][CW], ri[JT][CW], ir[JT][CW];
#pragma unroll
    for (int g = 0; g < KG; g++) Word<P>::template load<false>(pa[g], wi, va[g]);
    T y[JT][4][PW];
#pragma unroll
    for (int t = 0; t < JT; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (py[t][r]) Word<P>::template load<false>(py[t][r], wi, y[t][r]);
#pragma unroll
    for (int t = 0; t < JT; t++)
#pragma unroll
      for (int c = 0; c < CW; c++) rr[t][c] = ii[t][c] = ri[t][c] = ir[t][c] = zero_acc<Acc>();
#pragma unroll
    for (int g = 0; g < KG; g++)
#pragma unroll
      for (int c = 0; c < CW; c++) {
        const T ar = use[g] ? va[g][2 * c] : (T)0, ai = use[g] ? va[g][2 * c + 1] : (T)0;
#pragma unroll
        for (int t = 0; t < JT; t++) {
          rr[t][c] = M::mma(mr[g][t], ar, rr[t][c]);
          ri[t][c] = M::mma(mr[g][t], ai, ri[t][c]);
          ii[t][c] = M::mma(mi[g][t], ai, ii[t][c]);
          ir[t][c] = M::mma(mi[g][t], ar, ir[t][c]);
        }
      }
#pragma unroll
    for (int t = 0; t < JT; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (po[t][r]) {
          T o[PW];
#pragma unroll
          for (int c = 0; c < CW; c++) {
            o[2 * c] = rr[t][c][r] - ii[t][c][r];
            o[2 * c + 1] = ri[t][c][r] + ir[t][c][r];
          }
          if (py[t][r]) {
#pragma unroll
            for (int k = 0; k < PW; k++) o[k] = y[t][r][k] + o[k];
          }
          Word<P>::template store<false>(po[t][r], wi, o);
        }
  }
}

static long block_sites(const GeomDesc &g) { return (g.vh + 63) / 64 * 64; }
template <int P, int S> static int block_units(const GeomDesc &g) {
  return (int)((g.vh + kSiteBlock - 1) / kSiteBlock * (kSiteBlock / S) * words_of<P>(kSpinorReals));
}

template <int P, int IT, int JT>
static void gram_tiles(const GeomDesc &g, const BlockArgs &ba, bool same, int nunits, int grid, double *partials,
                       hipStream_t st) {
  if constexpr (IT == JT) {
    if (same) {
      k_block_gram<P, IT, JT, true><<<grid, kBlockThreads, 0, st>>>(ba, block_sites(g), nunits, partials);
      return;
    }
  }
  k_block_gram<P, IT, JT, false><<<grid, kBlockThreads, 0, st>>>(ba, block_sites(g), nunits, partials);
}
template <int P> static int gram_prec(const GeomDesc &g, const BlockArgs &ba, bool same, double *partials, hipStream_t st) {
  const int nunits = block_units<P, kGramSites>(g);
  const int want = (nunits + kBlockWaves - 1) / kBlockWaves, grid = want < kMaxGramBlocks ? want : kMaxGramBlocks;
  const bool i2 = ba.na > kGramTile, j2 = ba.nb > kGramTile;
  if (i2 && j2) gram_tiles<P, 2, 2>(g, ba, same, nunits, grid, partials, st);
  else if (i2) gram_tiles<P, 2, 1>(g, ba, same, nunits, grid, partials, st);
  else if (j2) gram_tiles<P, 1, 2>(g, ba, same, nunits, grid, partials, st);
  else gram_tiles<P, 1, 1>(g, ba, same, nunits, grid, partials, st);
  return grid;
}

hipError_t block_gram_launch(const GeomDesc &g, const BlockArgs &ba, double *partials, double *out, hipStream_t st) {
  if (ba.na < 1 || ba.nb < 1 || ba.na > kMaxRhs || ba.nb > kMaxRhs) return hipErrorInvalidValue;
  bool same = ba.na == ba.nb;
  for (int i = 0; i < ba.na && same; i++) same = ba.a[i] == ba.b[i];
  int grid;
  switch (g.prec) {
    case P64: grid = gram_prec<P64>(g, ba, same, partials, st); break;
    case P32: grid = gram_prec<P32>(g, ba, same, partials, st); break;
    default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int ne = ba.na * ba.nb * 2;
  if (same) k_block_gram_finalize<true><<<(ne + 15) / 16, 256, 0, st>>>(partials, grid, ba.na, ba.nb, out);
  else k_block_gram_finalize<false><<<(ne + 15) / 16, 256, 0, st>>>(partials, grid, ba.na, ba.nb, out);
  return hipGetLastError();
}

template <int P, int KG>
static void combine_groups(const GeomDesc &g, const BlockArgs &ba, int nunits, int grid, const double *mat,
                           hipStream_t st) {
  const long ns = block_sites(g);
  if (ba.nb > 16) k_block_combine<P, KG, 2><<<grid, kBlockThreads, 0, st>>>(ba, ns, nunits, mat);
  else k_block_combine<P, KG, 1><<<grid, kBlockThreads, 0, st>>>(ba, ns, nunits, mat);
}
template <int P> static void combine_prec(const GeomDesc &g, const BlockArgs &ba, const double *mat, hipStream_t st) {
  const int nunits = block_units<P, kCombineSites>(g);
  const int want = (nunits + kBlockWaves - 1) / kBlockWaves, grid = want < 2048 ? want : 2048;
  switch ((ba.na + 3) / 4) {
#define CG(K) \
  case K: combine_groups<P, K>(g, ba, nunits, grid, mat, st); break;
    CG(1) CG(2) CG(3) CG(4) CG(5) CG(6) CG(7) CG(8)
#undef CG
  }
}

hipError_t block_combine_launch(const GeomDesc &g, const BlockArgs &ba, const double *mat, hipStream_t st) {
  if (ba.na < 1 || ba.nb < 1 || ba.na > kMaxRhs || ba.nb > kMaxRhs) return hipErrorInvalidValue;
  switch (g.prec) {
    case P64: combine_prec<P64>(g, ba, mat, st); break;
    case P32: combine_prec<P32>(g, ba, mat, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace qphix_amd
