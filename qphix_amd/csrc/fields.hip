// Field preparation kernels: canonical <-> device layout packers, seeded gauge
// and spinor generation, clover term construction / inversion and precision
// conversion. These run once per configuration; they favour clarity over speed.
#include "fields.hpp"
#include "hop_impl.hpp"

namespace qphix_amd {

// ---------------------------------------------------------------------------
// canonical index helpers (QDP++ checkerboarded lexicographic order)
// ---------------------------------------------------------------------------
struct Lat {
  int L[4];
  int nxh;
  long vh;
};

__device__ inline void cb_coords(const Lat &l, int cb, long s, int c[4]) {
  long r = s;
  const int xh = (int)(r % l.nxh);
  r /= l.nxh;
  c[1] = (int)(r % l.L[1]);
  r /= l.L[1];
  c[2] = (int)(r % l.L[2]);
  c[3] = (int)(r / l.L[2]);
  c[0] = 2 * xh + ((c[1] + c[2] + c[3] + cb) & 1);
}
__device__ inline long cb_site(const Lat &l, const int c[4]) {
  return (((long)c[3] * l.L[2] + c[2]) * l.L[1] + c[1]) * l.nxh + c[0] / 2;
}
__device__ inline int cb_of(const int c[4]) { return (c[0] + c[1] + c[2] + c[3]) & 1; }

// ---------------------------------------------------------------------------
// spinor pack / unpack / generate / convert
// ---------------------------------------------------------------------------
template <int P>
__global__ void k_pack_spinor(void *dst, size_t vs, long vh, const double *src) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<P>::calc v[kSpinorReals];
  for (int k = 0; k < kSpinorReals; k++) v[k] = (typename PT<P>::calc)src[s * kSpinorReals + k];
  store_spinor<P>(dst, vs, s, v);
}

template <int P>
__global__ void k_unpack_spinor(double *dst, size_t vs, long vh, const void *src) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<P>::calc v[kSpinorReals];
  load_spinor<P>(src, vs, s, v);
  for (int k = 0; k < kSpinorReals; k++) dst[s * kSpinorReals + k] = (double)v[k];
}

__device__ inline uint64_t splitmix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}
__device__ inline double uniform01(uint64_t seed, uint64_t counter) {
  const uint64_t h = splitmix64(splitmix64(seed) ^ counter);
  return ((double)(h >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}
__device__ inline void gauss_pair(uint64_t seed, uint64_t counter, double &g0, double &g1) {
  const double u1 = uniform01(seed, 2 * counter), u2 = uniform01(seed, 2 * counter + 1);
  const double r = sqrt(-2.0 * log(u1));
  const double th = 6.283185307179586476925286766559 * u2;
  g0 = r * cos(th);
  g1 = r * sin(th);
}
constexpr uint64_t kTagGauge = 0x6761756765000000ULL;
constexpr uint64_t kTagSpinor = 0x7370696e6f720000ULL;

template <int P>
__global__ void k_gen_spinor(void *dst, size_t vs, Lat l, int cb, uint64_t seed) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= l.vh) return;
  int c[4];
  cb_coords(l, cb, s, c);
  const long lf = c[0] + (long)l.L[0] * (c[1] + (long)l.L[1] * (c[2] + (long)l.L[2] * c[3]));
  typename PT<P>::calc v[kSpinorReals];
  for (int k = 0; k < 12; k++) {
    double g0, g1;
    gauss_pair(seed ^ kTagSpinor, (uint64_t)lf * 12 + k, g0, g1);
    v[2 * k] = (typename PT<P>::calc)g0;
    v[2 * k + 1] = (typename PT<P>::calc)g1;
  }
  store_spinor<P>(dst, vs, s, v);
}

template <int PO, int PI>
__global__ void k_convert_spinor(void *out, const void *in, size_t vs, long vh, double scale) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<PI>::calc a[kSpinorReals];
  typename PT<PO>::calc b[kSpinorReals];
  load_spinor<PI>(in, vs, s, a);
  typedef typename PT<PO>::calc TO;
  const TO sc = (TO)scale;
  for (int k = 0; k < kSpinorReals; k++) b[k] = sc * (TO)a[k];
  store_spinor<PO>(out, vs, s, b);
}

// ---------------------------------------------------------------------------
// gauge
// ---------------------------------------------------------------------------
// canonical full gauge (double [V][4][18]) -> one checkerboard array
template <int P, bool C12>
__global__ void k_pack_gauge(void *dst, size_t vs, Lat l, int cb, const double *src) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= l.vh) return;
  constexpr int LR = C12 ? 12 : 18;
  typename PT<P>::calc v[8 * LR];
  int c[4];
  cb_coords(l, cb, s, c);
  const long self = cb * l.vh + s;
  for (int mu = 0; mu < 4; mu++) {
    int d[4] = {c[0], c[1], c[2], c[3]};
    d[mu] = (d[mu] - 1 + l.L[mu]) % l.L[mu];
    const long nb = (long)cb_of(d) * l.vh + cb_site(l, d);
    for (int k = 0; k < LR; k++) {
      v[(2 * mu) * LR + k] = (typename PT<P>::calc)src[(nb * 4 + mu) * 18 + k];
      v[(2 * mu + 1) * LR + k] = (typename PT<P>::calc)src[(self * 4 + mu) * 18 + k];
    }
  }
  store_all<P, words_of<P>(8 * LR)>(dst, vs, s, v);
}

// U_mu(x) = reunit(exp(i eps A)) into a canonical double gauge array
__global__ void k_gen_gauge(double *u, Lat l, uint64_t seed, double eps) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * l.vh) return;
  const int cb = (int)(i / l.vh);
  int c[4];
  cb_coords(l, cb, i - cb * l.vh, c);
  const long lf = c[0] + (long)l.L[0] * (c[1] + (long)l.L[1] * (c[2] + (long)l.L[2] * c[3]));
  for (int mu = 0; mu < 4; mu++) {
    cx<double> G[9], M[9], R[9], T[9], tmp[9];
    for (int k = 0; k < 9; k++) {
      double g0, g1;
      gauss_pair(seed ^ kTagGauge, (uint64_t)(lf * 4 + mu) * 9 + k, g0, g1);
      G[k] = mk(g0, g1);
    }
    double tr = G[0].r + G[4].r + G[8].r;
    double nrm = 0;
    for (int a = 0; a < 3; a++)
      for (int b = 0; b < 3; b++) {
        cx<double> h = scale(0.5, G[3 * a + b] + conj(G[3 * b + a]));
        if (a == b) h.r -= tr / 3.0;
        M[3 * a + b] = mk(-eps * h.i, eps * h.r);  // i * eps * A
        nrm += M[3 * a + b].r * M[3 * a + b].r + M[3 * a + b].i * M[3 * a + b].i;
      }
    nrm = sqrt(nrm);
    int sq = 0;
    while (nrm > 0.25) {
      nrm *= 0.5;
      sq++;
    }
    const double sc = ldexp(1.0, -sq);
    for (int k = 0; k < 9; k++) {
      M[k] = scale(sc, M[k]);
      R[k] = mk(k % 4 == 0 ? 1.0 : 0.0, 0.0);
      T[k] = R[k];
    }
    for (int n = 1; n <= 18; n++) {
      for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) tmp[3 * a + b] = T[3 * a] * M[b] + T[3 * a + 1] * M[3 + b] + T[3 * a + 2] * M[6 + b];
      for (int k = 0; k < 9; k++) {
        T[k] = scale(1.0 / n, tmp[k]);
        R[k] = R[k] + T[k];
      }
    }
    for (int q = 0; q < sq; q++) {
      for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) tmp[3 * a + b] = R[3 * a] * R[b] + R[3 * a + 1] * R[3 + b] + R[3 * a + 2] * R[6 + b];
      for (int k = 0; k < 9; k++) R[k] = tmp[k];
    }
    // reunitarise: row 0 normalised, row 1 orthonormalised, row 2 = conj(r0 x r1)
    double n0 = 0;
    for (int k = 0; k < 3; k++) n0 += R[k].r * R[k].r + R[k].i * R[k].i;
    n0 = 1.0 / sqrt(n0);
    for (int k = 0; k < 3; k++) R[k] = scale(n0, R[k]);
    cx<double> dd = mk(0.0, 0.0);
    for (int k = 0; k < 3; k++) dd = dd + cmulc(R[k], R[3 + k]);
    for (int k = 0; k < 3; k++) R[3 + k] = R[3 + k] - dd * R[k];
    double n1 = 0;
    for (int k = 0; k < 3; k++) n1 += R[3 + k].r * R[3 + k].r + R[3 + k].i * R[3 + k].i;
    n1 = 1.0 / sqrt(n1);
    for (int k = 0; k < 3; k++) R[3 + k] = scale(n1, R[3 + k]);
    for (int k = 0; k < 3; k++) {
      const int a = (k + 1) % 3, b = (k + 2) % 3;
      R[6 + k] = conj(R[a] * R[3 + b] - R[b] * R[3 + a]);
    }
    double *o = u + (i * 4 + mu) * 18;
    for (int k = 0; k < 9; k++) {
      o[2 * k] = R[k].r;
      o[2 * k + 1] = R[k].i;
    }
  }
}

template <int PO, int PI, bool CO, bool CI>
__global__ void k_convert_gauge(void *out, const void *in, size_t vs, long vh) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  constexpr int LI = CI ? 12 : 18, LO = CO ? 12 : 18;
  typename PT<PI>::calc a[8 * LI];
  typename PT<PO>::calc b[8 * LO];
  load_range<PI, words_of<PI>(8 * LI), 0, words_of<PI>(8 * LI)>(in, vs, s, a);
  for (int l = 0; l < 8; l++) {
    typedef typename PT<PI>::calc TI;
    cx<TI> U[3][3];
    make_link<CI>(a + l * LI, U);
    for (int r = 0; r < (CO ? 2 : 3); r++)
      for (int c = 0; c < 3; c++) {
        b[l * LO + (3 * r + c) * 2] = (typename PT<PO>::calc)U[r][c].r;
        b[l * LO + (3 * r + c) * 2 + 1] = (typename PT<PO>::calc)U[r][c].i;
      }
  }
  store_all<PO, words_of<PO>(8 * LO)>(out, vs, s, b);
}

// ---------------------------------------------------------------------------
// clover
// ---------------------------------------------------------------------------
// Chroma site record (diag[2][6], offd[2][15][2]) <-> per-block (diag[6], offd[15][2])
template <int P>
__global__ void k_pack_clover(void *dst, size_t vs, long vh, const double *src) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<P>::calc v[kCloverReals];
  const double *c = src + s * kCloverReals;
  for (int b = 0; b < 2; b++) {
    for (int k = 0; k < 6; k++) v[36 * b + k] = (typename PT<P>::calc)c[6 * b + k];
    for (int k = 0; k < 30; k++) v[36 * b + 6 + k] = (typename PT<P>::calc)c[12 + 30 * b + k];
  }
  store_all<P, words_of<P>(kCloverReals)>(dst, vs, s, v);
}
template <int P>
__global__ void k_unpack_clover(double *dst, size_t vs, long vh, const void *src) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<P>::calc v[kCloverReals];
  load_range<P, words_of<P>(kCloverReals), 0, words_of<P>(kCloverReals)>(src, vs, s, v);
  double *c = dst + s * kCloverReals;
  for (int b = 0; b < 2; b++) {
    for (int k = 0; k < 6; k++) c[6 * b + k] = (double)v[36 * b + k];
    for (int k = 0; k < 30; k++) c[12 + 30 * b + k] = (double)v[36 * b + 6 + k];
  }
}
template <int P>
__global__ void k_pack_full_clover(void *dst, size_t vs, long vh, const double *src) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<P>::calc v[kFullCloverReals];
  for (int k = 0; k < kFullCloverReals; k++) v[k] = (typename PT<P>::calc)src[s * kFullCloverReals + k];
  store_all<P, words_of<P>(kFullCloverReals)>(dst, vs, s, v);
}
template <int PO, int PI, int N>
__global__ void k_convert_words(void *out, const void *in, size_t vs, long vh) {
  const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= vh) return;
  typename PT<PI>::calc a[N];
  typename PT<PO>::calc b[N];
  load_range<PI, words_of<PI>(N), 0, words_of<PI>(N)>(in, vs, s, a);
  for (int k = 0; k < N; k++) b[k] = (typename PT<PO>::calc)a[k];
  store_all<PO, words_of<PO>(N)>(out, vs, s, b);
}

typedef cx<double> zd;

// ---------------------------------------------------------------------------
// clover term: one kernel from the links to the stored blocks.
//
// A work-group of two wavefronts takes 64 sites: each wavefront computes three
// of the six planes of the field strength of its lane's site and leaves their
// nine reals (F is anti-Hermitian) in LDS; after a barrier wavefront b builds
// chiral block b from them, inverts it where asked and stores it in the field
// precision. Nothing but the links is read and nothing but the result is
// written. Bound: the 96 link reads a site (12 distinct ones a plane), most of
// them from beyond the L2, whose 4 MB cannot hold the t neighbours of the
// 8192 sites an XCD has in flight; the FP64 products are a third of the time
// (as FMA chains, a third fewer instructions, they gave 1%, not kept). The
// work-groups of an XCD walk one contiguous range (551 us without that).
// Measured at 24^3x48, FP64, A^-1: 467 us a build; the form before, eight
// kernels per 2^20 sites through 252 doubles of scratch a site, took 772 us
// of kernels and 19 ms with the scratch allocated and freed by each build.
// ---------------------------------------------------------------------------

// U_mu at a site: link 2 mu + 1 of its record. The link's place within its
// first word is the same for every mu (2 mu + 1 is odd), so mu may be a
// run-time value. load() reads the words that hold it, make() rebuilds it.
template <int P, bool C12> struct SiteLink {
  typedef GaugeLayout<P, C12> GL;
  typedef typename PT<P>::calc T;
  static constexpr int pw = PT<P>::per_word;
  static constexpr int off = GL::link_reals % pw;
  static constexpr int w0 = GL::link_reals / pw;
  static constexpr int nwl = (off + GL::link_reals + pw - 1) / pw;
  T buf[nwl * pw];
  __device__ inline void load(const void *u, size_t vs, int mu, unsigned s) {
#pragma unroll
    for (int w = 0; w < nwl; w++)
      Word<P>::template load<false>(u, widx(s, w0 + mu * GL::pair_words + w, GL::nw), buf + w * pw);
    if constexpr (PT<P>::scaled) {
      const T sc = site_scale<P>(u, vs, s, GL::nw);
#pragma unroll
      for (int k = 0; k < nwl * pw; k++) buf[k] *= sc;
    }
  }
  __device__ inline void make(zd (&U)[3][3]) const {
    cx<T> Ut[3][3];
    make_link<C12>(buf + off, Ut);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) U[a][b] = mk((double)Ut[a][b].r, (double)Ut[a][b].i);
  }
};

// a site of the full lattice: coordinates, checkerboard site and checkerboard
struct CloverSite {
  int c0, c1, c2, c3;
};
__device__ inline int wrapped(int c, int d, int n) {
  c += d;
  return c < 0 ? c + n : c >= n ? c - n : c;
}
__device__ inline void shift(CloverSite &x, const Lat &l, int mu, int d) {
  if (mu == 0) x.c0 = wrapped(x.c0, d, l.L[0]);
  else if (mu == 1) x.c1 = wrapped(x.c1, d, l.L[1]);
  else if (mu == 2) x.c2 = wrapped(x.c2, d, l.L[2]);
  else x.c3 = wrapped(x.c3, d, l.L[3]);
}

// X = X U, or X U^+ (DAG)
template <bool DAG> __device__ inline void times_link(zd (&X)[3][3], const zd (&U)[3][3]) {
  zd Y[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      zd t = mk(0.0, 0.0);
#pragma unroll
      for (int k = 0; k < 3; k++) t = t + X[a][k] * (DAG ? conj(U[b][k]) : U[k][b]);
      Y[a][b] = t;
    }
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) X[a][b] = Y[a][b];
}

constexpr int kCloverSites = 64;  // sites per work-group
constexpr int kPlaneReals = 9;    // reals of an anti-Hermitian 3x3 matrix

// coef * F_{mu nu}(x) = coef * (Q - Q^+) / 8, Q the sum of the four clover
// leaves at x (tests/mesfield.cc:24-64); its diagonal (imaginary) in
// F[0..2], (1,0), (2,0), (2,1) in F[3..8], entry e of lane j at F[e * 64 + j].
// Leaf q walks the plaquette's four steps +mu +nu -mu -nu from step q on, so
// the sixteen factors are one loop: unrolled, the compiler kept the twelve
// distinct links live (512 registers and a spill); rolled, with the next
// link's load ahead of the product, it fits two wavefronts per SIMD.
template <int P, bool C12>
__device__ inline void field_strength(const void *u0, const void *u1, size_t vs, const Lat &l, const CloverSite &x,
                                      int mu, int nu, double coef, double *F) {
  zd Q[3][3], X[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) Q[a][b] = X[a][b] = mk(0.0, 0.0);
  CloverSite pos = x;
  SiteLink<P, C12> link;
  // the link of factor n (a step against its direction takes the link of the
  // site it leads to), and the step
  auto fetch = [&](int n) {
    if ((n & 3) == 0) pos = x;
    const int k = ((n >> 2) + n) & 3, dir = (k & 1) ? nu : mu;
    if (k >> 1) shift(pos, l, dir, -1);
    const unsigned s = (((unsigned)pos.c3 * l.L[2] + pos.c2) * l.L[1] + pos.c1) * l.nxh + ((unsigned)pos.c0 >> 1);
    link.load(((pos.c0 + pos.c1 + pos.c2 + pos.c3) & 1) ? u1 : u0, vs, dir, s);
    if (!(k >> 1)) shift(pos, l, dir, 1);
  };
  fetch(0);
#pragma nounroll
  for (int n = 0; n < 16; n++) {
    zd U[3][3];
    link.make(U);
    if (n < 15) fetch(n + 1);
    const bool dag = (((n >> 2) + n) & 2) != 0;
    if ((n & 3) == 0) {
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) X[a][b] = dag ? conj(U[b][a]) : U[a][b];
    } else if (dag) {
      times_link<true>(X, U);
    } else {
      times_link<false>(X, U);
    }
    if ((n & 3) == 3) {
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) Q[a][b] = Q[a][b] + X[a][b];
    }
  }
  const double f = 0.125 * coef;
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b <= a; b++) {
      const zd v = scale(f, Q[a][b] - conj(Q[b][a]));
      if (a == b) {
        F[a * kCloverSites] = v.i;
      } else {
        F[(3 + 2 * (a + b - 1)) * kCloverSites] = v.r;
        F[(4 + 2 * (a + b - 1)) * kCloverSites] = v.i;
      }
    }
}

// lower-triangle storage of a Hermitian 6x6 matrix: (i, j), i >= j
__host__ __device__ constexpr int tri(int i, int j) { return i * (i + 1) / 2 + j; }
__device__ inline zd hel(const zd (&M)[21], int i, int j) { return i >= j ? M[tri(i, j)] : conj(M[tri(j, i)]); }

// entry (a, b) of plane k of the field strength from the lane's LDS column
__device__ inline zd fplane(const double *F, int k, int a, int b) {
  const double *p = F + k * kPlaneReals * kCloverSites;
  if (a == b) return mk(0.0, p[a * kCloverSites]);
  const double re = p[(3 + 2 * (a + b - 1)) * kCloverSites], im = p[(4 + 2 * (a + b - 1)) * kCloverSites];
  return a > b ? mk(re, im) : mk(-re, im);
}

// chiral block b of the clover term in Chroma's packing
// (tests/clover_term_qdp_w.h:325-442), index i = 3 * (spin - 2b) + colour:
// with s = +1 (b = 0) or -1 (b = 1), G = i (F01 - s F23), H = (i F12 - F02) - s (i F03 + F13)
//   A_b = [[diag_mass + G, H^+], [H, diag_mass - G]]
// (F already carries the plane's clover coefficient)
__device__ inline void clover_block(const double *F, int blk, double dm, zd (&A)[21]) {
  const double s = blk == 0 ? 1.0 : -1.0;
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b <= a; b++) {
      const zd d = fplane(F, 0, a, b) - scale(s, fplane(F, 5, a, b));
      const zd g = mk(-d.i, d.r);
      A[tri(a, b)] = a == b ? mk(dm + g.r, 0.0) : g;
      A[tri(a + 3, b + 3)] = a == b ? mk(dm - g.r, 0.0) : scale(-1.0, g);
    }
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      const zd f2 = fplane(F, 2, a, b), f3 = fplane(F, 3, a, b);
      const zd em = mk(-f2.i, f2.r) + fplane(F, 4, a, b);
      const zd bm = mk(-f3.i, f3.r) - fplane(F, 1, a, b);
      A[tri(a + 3, b)] = bm - scale(s, em);
    }
}

// M <- M^-1 for Hermitian positive definite M: Cholesky M = L L^+ in place,
// Li = L^-1 by forward substitution, M^-1 = Li^+ Li
__device__ inline void hpd_inverse(zd (&M)[21]) {
  double dinv[6];
#pragma unroll
  for (int c = 0; c < 6; c++) {
    double d = M[tri(c, c)].r;
#pragma unroll
    for (int k = 0; k < c; k++) d -= M[tri(c, k)].r * M[tri(c, k)].r + M[tri(c, k)].i * M[tri(c, k)].i;
    d = sqrt(d);
    dinv[c] = 1.0 / d;
    M[tri(c, c)] = mk(d, 0.0);
#pragma unroll
    for (int i = c + 1; i < 6; i++) {
      zd t = M[tri(i, c)];
#pragma unroll
      for (int k = 0; k < c; k++) t = t - M[tri(i, k)] * conj(M[tri(c, k)]);
      M[tri(i, c)] = scale(dinv[c], t);
    }
  }
  zd Li[21];
#pragma unroll
  for (int c = 0; c < 6; c++) {
    Li[tri(c, c)] = mk(dinv[c], 0.0);
#pragma unroll
    for (int i = c + 1; i < 6; i++) {
      zd t = mk(0.0, 0.0);
#pragma unroll
      for (int k = c; k < i; k++) t = t + M[tri(i, k)] * Li[tri(k, c)];
      Li[tri(i, c)] = scale(-dinv[i], t);
    }
  }
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int j = 0; j <= i; j++) {
      zd t = mk(0.0, 0.0);
#pragma unroll
      for (int k = i; k < 6; k++) t = t + cmulc(Li[tri(k, i)], Li[tri(k, j)]);
      M[tri(i, j)] = t;
    }
}

// A <- A A + shift
__device__ inline void square_shift(zd (&A)[21], double shift) {
  zd S[21];
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int j = 0; j <= i; j++) {
      zd t = mk(i == j ? shift : 0.0, 0.0);
#pragma unroll
      for (int q = 0; q < 6; q++) t = t + hel(A, i, q) * hel(A, q, j);
      S[tri(i, j)] = t;
    }
#pragma unroll
  for (int k = 0; k < 21; k++) A[k] = S[k];
}

constexpr bool clover_full(int what) { return what == 2 || what == 3 || what == 4; }

// what: 0 A, 1 A^-1, 5 eps (A^2 + mu^2 - eps^2)^-1 (packed Hermitian, 36
// reals per block); 2 (A + i mu g5)^-1 = (A^2 + mu^2)^-1 (A - i mu g5),
// 3 (A^2 + mu^2 - eps^2)^-1 (A - i mu g5), 4 the same with + i mu g5 (full
// complex blocks, 72 reals per block); o(e, value) takes the reals of block blk
template <int WHAT, typename Out>
__device__ inline void clover_result(const double *F, int blk, double dm, double mu, double eps, Out o) {
  zd A[21];
  clover_block(F, blk, dm, A);
  if constexpr (!clover_full(WHAT)) {
    if constexpr (WHAT == 1) hpd_inverse(A);
    if constexpr (WHAT == 5) {
      square_shift(A, mu * mu - eps * eps);
      hpd_inverse(A);
#pragma unroll
      for (int k = 0; k < 21; k++) A[k] = scale(eps, A[k]);
    }
#pragma unroll
    for (int i = 0; i < 6; i++) o(i, A[tri(i, i)].r);
#pragma unroll
    for (int i = 1; i < 6; i++)
#pragma unroll
      for (int k = 0; k < i; k++) {
        const int e = i * (i - 1) / 2 + k;
        o(6 + 2 * e, A[tri(i, k)].r);
        o(6 + 2 * e + 1, A[tri(i, k)].i);
      }
  } else {
    square_shift(A, WHAT == 2 ? mu * mu : mu * mu - eps * eps);
    hpd_inverse(A);  // A now holds N = (A^2 + shift)^-1
    zd B[21];
    clover_block(F, blk, dm, B);  // the block again, for the factor on the right
    const double g5 = blk == 0 ? 1.0 : -1.0;
    const double tw = (WHAT == 4 ? 1.0 : -1.0) * g5 * mu;
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
      for (int k = 0; k < 6; k++) {
        zd t = mk(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < 6; q++) t = t + hel(A, i, q) * hel(B, q, k);
        const zd nik = hel(A, i, k);
        t = t + mk(-tw * nik.i, tw * nik.r);
        o(12 * i + 2 * k, t.r);
        o(12 * i + 2 * k + 1, t.i);
      }
  }
}

// coef of plane 01 02 03 12 13 23: the planes with t take the temporal one
template <int P, bool C12, int WHAT>
__global__ void __launch_bounds__(2 * kCloverSites, 2) k_clover(const void *u0, const void *u1, size_t vs, Lat l, int cb,
                                                             double cr, double ct, double dm, double mu, double eps,
                                                             void *out) {
  typedef typename PT<P>::calc T;
  constexpr int N = clover_full(WHAT) ? kFullCloverReals : kCloverReals;  // reals per site
  constexpr int pw = PT<P>::per_word, nw = N / pw;
  // the half precisions scale a site's values by the largest of both blocks
  // and pack eight to a word, so their blocks meet in LDS before the store
  constexpr int kFBytes = 6 * kPlaneReals * kCloverSites * 8;
  constexpr int kVBytes = PT<P>::scaled ? N * kCloverSites * 4 : 0;
  __shared__ double lds[(kFBytes > kVBytes ? kFBytes : kVBytes) / 8];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const long s = (long)xcd_block() * kCloverSites + lane;
  const bool live = s < l.vh;
  double *F = lds + lane;
  if (live) {
    CloverSite x;
    unsigned r = (unsigned)s;
    const unsigned xh = r % (unsigned)l.nxh;
    r /= (unsigned)l.nxh;
    x.c1 = (int)(r % (unsigned)l.L[1]);
    r /= (unsigned)l.L[1];
    x.c2 = (int)(r % (unsigned)l.L[2]);
    x.c3 = (int)(r / (unsigned)l.L[2]);
    x.c0 = 2 * (int)xh + ((x.c1 + x.c2 + x.c3 + cb) & 1);
#pragma nounroll
    for (int k = 3 * wave; k < 3 * wave + 3; k++) {
      const int pm = k < 3 ? 0 : k < 5 ? 1 : 2, pn = k < 3 ? k + 1 : k < 5 ? k - 1 : 3;
      field_strength<P, C12>(u0, u1, vs, l, x, pm, pn, pn == 3 ? ct : cr, F + k * kPlaneReals * kCloverSites);
    }
  }
  __syncthreads();
  if constexpr (!PT<P>::scaled) {
    if (!live) return;
    T v[N / 2];
    clover_result<WHAT>(F, wave, dm, mu, eps, [&](int e, double x) { v[e] = (T)x; });
#pragma unroll
    for (int w = 0; w < nw / 2; w++) Word<P>::template store<false>(out, widx(s, wave * (nw / 2) + w, nw), v + w * pw);
  } else {
    float v[N / 2];
    if (live) clover_result<WHAT>(F, wave, dm, mu, eps, [&](int e, double x) { v[e] = (float)x; });
    __syncthreads();  // F is done with
    float *V = reinterpret_cast<float *>(lds) + lane;
    if (live) {
#pragma unroll
      for (int e = 0; e < N / 2; e++) V[(wave * (N / 2) + e) * kCloverSites] = v[e];
    }
    __syncthreads();
    if (!live) return;
    float m = 0.f;
    for (int e = 0; e < N; e++) m = fmaxf(m, fabsf(V[e * kCloverSites]));
    const float inv = m > 0.f ? 1.0f / m : 0.f;
    if (wave == 0) reinterpret_cast<float *>(reinterpret_cast<char *>(out) + (size_t)nw * vs * 16)[s] = m;
    for (int w = wave; w < nw; w += 2) {
      float t[pw];
#pragma unroll
      for (int k = 0; k < pw; k++) t[k] = V[(w * pw + k) * kCloverSites] * inv;
      Word<P>::template store<false>(out, widx(s, w, nw), t);
    }
  }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
static inline dim3 grid_for(long n, int b = 256) { return dim3((unsigned)((n + b - 1) / b)); }
static inline Lat make_lat(const GeomDesc &g) {
  Lat l;
  for (int k = 0; k < 4; k++) l.L[k] = g.L[k];
  l.nxh = g.L[0] / 2;
  l.vh = g.vh;
  return l;
}

#define PREC_SWITCH(p, F) \
  switch (p) {            \
    case P64: { constexpr int PP = P64; F; } break; \
    case P32: { constexpr int PP = P32; F; } break; \
    case P16: { constexpr int PP = P16; F; } break; \
    case PB16: { constexpr int PP = PB16; F; } break; \
    default: return hipErrorInvalidValue; \
  }

hipError_t fld_pack_spinor(const GeomDesc &g, void *dst, const double *dsrc, hipStream_t st) {
  PREC_SWITCH(g.prec, (k_pack_spinor<PP><<<grid_for(g.vh), 256, 0, st>>>(dst, g.vs, g.vh, dsrc)));
  return hipGetLastError();
}
hipError_t fld_unpack_spinor(const GeomDesc &g, double *ddst, const void *src, hipStream_t st) {
  PREC_SWITCH(g.prec, (k_unpack_spinor<PP><<<grid_for(g.vh), 256, 0, st>>>(ddst, g.vs, g.vh, src)));
  return hipGetLastError();
}
hipError_t fld_gen_spinor(const GeomDesc &g, void *dst, uint64_t seed, int cb, hipStream_t st) {
  Lat l = make_lat(g);
  PREC_SWITCH(g.prec, (k_gen_spinor<PP><<<grid_for(g.vh), 256, 0, st>>>(dst, g.vs, l, cb, seed)));
  return hipGetLastError();
}

template <int PO>
static hipError_t conv_spinor_in(int pin, void *out, const void *in, size_t vs, long vh, double scale, hipStream_t st) {
  switch (pin) {
    case P64: k_convert_spinor<PO, P64><<<grid_for(vh), 256, 0, st>>>(out, in, vs, vh, scale); break;
    case P32: k_convert_spinor<PO, P32><<<grid_for(vh), 256, 0, st>>>(out, in, vs, vh, scale); break;
    case P16: k_convert_spinor<PO, P16><<<grid_for(vh), 256, 0, st>>>(out, in, vs, vh, scale); break;
    case PB16: k_convert_spinor<PO, PB16><<<grid_for(vh), 256, 0, st>>>(out, in, vs, vh, scale); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t fld_convert_spinor(const GeomDesc &go, void *out, double scale, const GeomDesc &gi, const void *in,
                              hipStream_t st) {
  PREC_SWITCH(go.prec, return conv_spinor_in<PP>(gi.prec, out, in, go.vs, go.vh, scale, st));
  return hipSuccess;
}

hipError_t fld_pack_gauge_cb(const GeomDesc &g, void *dst, int cb, const double *dsrc, hipStream_t st) {
  Lat l = make_lat(g);
  if (g.c12) {
    PREC_SWITCH(g.prec, (k_pack_gauge<PP, true><<<grid_for(g.vh), 256, 0, st>>>(dst, g.vs, l, cb, dsrc)));
  } else {
    switch (g.prec) {
      case P64: k_pack_gauge<P64, false><<<grid_for(g.vh), 256, 0, st>>>(dst, g.vs, l, cb, dsrc); break;
      case P32: k_pack_gauge<P32, false><<<grid_for(g.vh), 256, 0, st>>>(dst, g.vs, l, cb, dsrc); break;
      default: return hipErrorInvalidValue;
    }
  }
  return hipGetLastError();
}
hipError_t fld_gen_gauge_canonical(const GeomDesc &g, double *du, uint64_t seed, double eps, hipStream_t st) {
  Lat l = make_lat(g);
  k_gen_gauge<<<grid_for(2 * g.vh, 128), 128, 0, st>>>(du, l, seed, eps);
  return hipGetLastError();
}

template <int PO, bool CO>
static hipError_t conv_gauge_in(const GeomDesc &gi, void *out, const void *in, size_t vs, long vh, hipStream_t st) {
  const dim3 gr = grid_for(vh, 128);
  if (gi.c12) {
    switch (gi.prec) {
      case P64: k_convert_gauge<PO, P64, CO, true><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
      case P32: k_convert_gauge<PO, P32, CO, true><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
      case P16: k_convert_gauge<PO, P16, CO, true><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
      case PB16: k_convert_gauge<PO, PB16, CO, true><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
      default: return hipErrorInvalidValue;
    }
  } else {
    switch (gi.prec) {
      case P64: k_convert_gauge<PO, P64, CO, false><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
      case P32: k_convert_gauge<PO, P32, CO, false><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
      default: return hipErrorInvalidValue;
    }
  }
  return hipGetLastError();
}
hipError_t fld_convert_gauge(const GeomDesc &go, void *out, const GeomDesc &gi, const void *in, hipStream_t st) {
  if (go.c12) {
    PREC_SWITCH(go.prec, return (conv_gauge_in<PP, true>(gi, out, in, go.vs, go.vh, st)));
  } else {
    switch (go.prec) {
      case P64: return conv_gauge_in<P64, false>(gi, out, in, go.vs, go.vh, st);
      case P32: return conv_gauge_in<P32, false>(gi, out, in, go.vs, go.vh, st);
      default: return hipErrorInvalidValue;
    }
  }
  return hipSuccess;
}

hipError_t fld_pack_clover(const GeomDesc &g, void *dst, const double *dsrc, hipStream_t st) {
  PREC_SWITCH(g.prec, (k_pack_clover<PP><<<grid_for(g.vh), 256, 0, st>>>(dst, g.vs, g.vh, dsrc)));
  return hipGetLastError();
}
hipError_t fld_unpack_clover(const GeomDesc &g, double *ddst, const void *src, hipStream_t st) {
  PREC_SWITCH(g.prec, (k_unpack_clover<PP><<<grid_for(g.vh), 256, 0, st>>>(ddst, g.vs, g.vh, src)));
  return hipGetLastError();
}
hipError_t fld_pack_full_clover(const GeomDesc &g, void *dst, const double *dsrc, hipStream_t st) {
  PREC_SWITCH(g.prec, (k_pack_full_clover<PP><<<grid_for(g.vh, 128), 128, 0, st>>>(dst, g.vs, g.vh, dsrc)));
  return hipGetLastError();
}

template <int PO, int N>
static hipError_t conv_words_in(int pin, void *out, const void *in, size_t vs, long vh, hipStream_t st) {
  const dim3 gr = grid_for(vh, 128);
  switch (pin) {
    case P64: k_convert_words<PO, P64, N><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
    case P32: k_convert_words<PO, P32, N><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
    case P16: k_convert_words<PO, P16, N><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
    case PB16: k_convert_words<PO, PB16, N><<<gr, 128, 0, st>>>(out, in, vs, vh); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t fld_convert_clover(const GeomDesc &go, void *out, const GeomDesc &gi, const void *in, int full,
                              hipStream_t st) {
  if (full) {
    PREC_SWITCH(go.prec, return (conv_words_in<PP, kFullCloverReals>(gi.prec, out, in, go.vs, go.vh, st)));
  } else {
    PREC_SWITCH(go.prec, return (conv_words_in<PP, kCloverReals>(gi.prec, out, in, go.vs, go.vh, st)));
  }
  return hipSuccess;
}

template <int P, bool C12>
static hipError_t clover_build_po(const GeomDesc &g, const void *u0, const void *u1, double cr, double ct, double dm,
                                  int cb, int what, double mu, double eps, void *out, hipStream_t st) {
  const Lat l = make_lat(g);
  const dim3 grid = grid_for(g.vh, kCloverSites);
  switch (what) {
#define CK(W) \
  case W: k_clover<P, C12, W><<<grid, 2 * kCloverSites, 0, st>>>(u0, u1, g.vs, l, cb, cr, ct, dm, mu, eps, out); break;
    CK(0) CK(1) CK(2) CK(3) CK(4) CK(5)
#undef CK
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// one launch, stream-ordered: no scratch, allocation or synchronisation
hipError_t fld_clover_build(const GeomDesc &g, const void *u0, const void *u1, double cr, double ct, double dm,
                            int cb, int what, double mu, double eps, void *out, hipStream_t st) {
  if (g.c12) {
    PREC_SWITCH(g.prec, return (clover_build_po<PP, true>(g, u0, u1, cr, ct, dm, cb, what, mu, eps, out, st)));
  } else {
    switch (g.prec) {
      case P64: return clover_build_po<P64, false>(g, u0, u1, cr, ct, dm, cb, what, mu, eps, out, st);
      case P32: return clover_build_po<P32, false>(g, u0, u1, cr, ct, dm, cb, what, mu, eps, out, st);
      default: return hipErrorInvalidValue;
    }
  }
  return hipSuccess;
}

}  // namespace qphix_amd
