// Products of the FP64 form on half of the G sphere.
//
// At the Gamma point a super wave psi = c1 + i c2 carries two real bands,
// c(-G) = conj(c(G)), and the projectors of a radial PRO table satisfy
// P(-G) = conj(P(G)).  With s = psi(G) + psi(-G) and d = psi(G) - psi(-G) the
// real bands are 2 c1 = (s.re, d.im), 2 c2 = (s.im, -d.re), so every product
// of a CP step is a real product over the (re, im) pairs of one G of each
// pair (G, -G): half the flops of the complex product over the whole sphere
// (8 M NBH NG -> 4 M NBH NG), and each projector value is formed once for
// both.  The half list (plan: hg) follows the sphere's order; equal |G|^2 are
// sorted by the integer components, so the partners -G of consecutive G are
// consecutive in reverse and both loads are coalesced.
//
// FP64 MFMA bound: 3.5 GFLOP per projector product at Si64 (512 projectors,
// 144 bands, 23 847 G) is 48 us at the rate of a large FP64 product.  Measured
// there against the complex products over the whole sphere: projections 287
// -> 77 us, ADDPRO 328 -> 99, forces 272 -> 85, the three band overlaps of a
// step 327 -> 85, ADDOPSI 101 -> 36.  The rest is the staging between the MFMAs:
// counted there, the matrix units are busy 63 % of the time in the projections,
// 56 in the overlaps, 58 in the forces, 51 in ADDPRO and 43 in ADDOPSI, and vector
// instructions take 11 to 20 %.  With selects on every load, 64-bit products in
// the addresses and (-i)^l by a switch the same kernels took 88, 107, 96, 89 and
// 39 us, with matrix units busy 42 to 58 % and vector instructions 14 to 24.
#include <algorithm>

#include "pw_device.h"

namespace {

constexpr int HK = 8;        // G pairs of a K chunk of the row products (16 real K)
constexpr int HKR = 2 * HK;  // real K of a staged chunk

// LDS row stride (doubles) of a staged operand: == 17 (mod 32), so that both
// the MFMA operand reads (16 consecutive columns of one row) and the staging
// stores (one column, rows hh) spread over the banks
constexpr int hpad(int w) { return w + ((17 - w % 32) + 32) % 32; }

// Projector factors on the half list, P(i,h) = (-i)^(l mod 2) F(k,h) E(atom,h);
// F carries the sign of the even power, (-1)^(l/2)
struct HalfP {
  const double *f;     // [NSP*LMNXX][NHP]
  const double2 *e;    // [NAT][NHP]
  const int4 *tab;     // per projector: offsets of its F and E rows, l mod 2, 0
  int npro, nhp;
  __device__ const double *frow(int4 t) const { return f + (unsigned)t.x; }
  __device__ const double2 *erow(int4 t) const { return e + (unsigned)t.y; }
};
// z (-i)^odd
__device__ inline double2 rot_odd(double2 z, int odd) {
  return make_double2(odd ? z.y : z.x, odd ? -z.x : z.y);
}

__global__ void k_half_f(ProjGeo q, int nsp, int nh, int nhp, const int2 *__restrict__ hg, double *f) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)nsp * q.lmnxx * nhp) return;
  const int k = (int)(idx / nhp), h = (int)(idx % nhp);
  const int isp = k / q.lmnxx, lmn = k % q.lmnxx;
  double v = 0.0;
  if (h < nh && lmn < q.lmnx[isp]) {
    const int ig = hg[h].x;
    v = q.ylm[(size_t)q.lmn_lm[k] * q.ngl + ig] * q.pro[(size_t)(q.ibpro[isp] + q.lmn_ln[k]) * q.ngl + ig];
    if (q.lmn_l[k] & 2) v = -v;
  }
  f[idx] = v;
}

__global__ void k_half_e(ProjGeo q, int nh, int nhp, const int2 *__restrict__ hg, double2 *e) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)q.nat * nhp) return;
  const int atom = (int)(idx / nhp), h = (int)(idx % nhp);
  e[idx] = h < nh ? eigr_of(q, atom, hg[h].x) : czero();
}

// psi of one super band at (G, -G).  The loads are unconditional (clamped
// indices): what is out of range meets a zero of the other operand or enters
// elements that are not written.  On these kernels every vector instruction
// counts: what the staging lost of them the kernels lost in time (figures above).
struct Pair {
  double2 p, m;
};
__device__ inline void load_pair(const double2 *__restrict__ psi, size_t off, int2 g, Pair &v) {
  v.p = psi[off + g.x];
  v.m = psi[off + g.y];
}
// the rows (re, im) of the two real bands: a = 2 c1, b = 2 c2; at the self pair
// G = 0 twice that, which the other operand makes good
struct Bands2 {
  double are, aim, bre, bim;
};
__device__ inline Bands2 split_pair(const Pair &v) {
  Bands2 r;
  r.are = v.p.x + v.m.x;
  r.bre = v.p.y + v.m.y;
  r.aim = v.p.y - v.m.y;
  r.bim = v.m.x - v.p.x;
  return r;
}

// ---------------------------------------------------------------------------
// Row products: part[split][r][n] = sum over the split's G pairs of A(r, re/im)
// X(n, re/im), n the real bands of psi.  A: projectors (PROJECTIONS) or the
// real bands of a second set (OVERLAP).
// ---------------------------------------------------------------------------
// A rows of a workgroup: 16 NW projectors, two (row, hh) per thread
template <int NW>
struct RowsP {
  HalfP p;
  __device__ void job(int) {}
  struct Row {
    const double *f[2];
    const double2 *e[2];
    int odd[2];
  };
  struct Pre {
    double f[2];
    double2 e[2];
  };
  __device__ void init(Row &w, int r0) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = r0 + (threadIdx.x >> 3) + 8 * NW * i;
      const int4 t = p.tab[min(r, p.npro - 1)];
      w.f[i] = p.frow(t);
      w.e[i] = p.erow(t);
      w.odd[i] = t.z;
    }
  }
  // h < NHP: the tables are zero beyond NH
  __device__ void fetch(const Row &w, int h, int2, Pre &v) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      v.f[i] = w.f[i][h];
      v.e[i] = w.e[i][h];
    }
  }
  template <int SA>
  __device__ void store(const Row &w, const Pre &v, bool self, bool, double (*sA)[SA]) const {
    const int hh = threadIdx.x & 7;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = (threadIdx.x >> 3) + 8 * NW * i;
      const double s = self ? 0.5 * v.f[i] : v.f[i];
      const double2 z = rot_odd(make_double2(s * v.e[i].x, s * v.e[i].y), w.odd[i]);
      sA[hh][r] = z.x;
      sA[HK + hh][r] = z.y;
    }
  }
};

// 16 NW real bands of psi (8 NW super bands), one (super band, hh) per
// thread; the G = 0 term counts twice (both operands hold twice their bands
// there, hence the half): sum over the pairs of A X is then 2 sum over the
// sphere of conj(c) c'.  Zero beyond the split's pairs.
template <int NW>
struct RowsX {
  const double2 *psis[kOvlJobs];
  int ngl, nbh;
  const double2 *psi;
  __device__ void job(int j) { psi = psis[j]; }
  struct Row {
    size_t off;
  };
  struct Pre {
    Pair v;
  };
  __device__ void init(Row &w, int r0) const {
    w.off = (size_t)min(r0 / 2 + (int)(threadIdx.x >> 3), nbh - 1) * ngl;
  }
  __device__ void fetch(const Row &w, int, int2 g, Pre &p) const { load_pair(psi, w.off, g, p.v); }
  template <int SA>
  __device__ void store(const Row &, const Pre &p, bool self, bool in, double (*sA)[SA]) const {
    const int hh = threadIdx.x & 7, n = 2 * (threadIdx.x >> 3);
    const Bands2 r = split_pair(p.v);
    const double w = in ? (self ? 0.5 : 1.0) : 0.0;
    sA[hh][n] = w * r.are;
    sA[hh][n + 1] = w * r.bre;
    sA[HK + hh][n] = w * r.aim;
    sA[HK + hh][n + 1] = w * r.bim;
  }
};

// the band operands of up to kOvlJobs products of one launch
struct HalfBands {
  const double2 *psi[kOvlJobs];
  int n;
};

// Workgroup: NW waves, 16 rows each, NC blocks of 16 real bands; K chunks of
// 16 double-buffered in LDS with one barrier each, the operands of the next
// chunk loaded into registers before the current chunk's MFMAs and stored
// after them.
template <class Rows, int NC, int NW>
__global__ void __launch_bounds__(64 * NW, 2) k_half_row(Rows rows, HalfBands bands,
                                                         const int2 *__restrict__ hg, int nh, int nrow, int ngl,
                                                         int nbh, int hsplit, int tr, int tb, int ns,
                                                         double *__restrict__ part) {
  constexpr int WR = 16 * NW, SA = hpad(WR), WC = 16 * NC, SB = hpad(WC);
  constexpr int NBT = (NC + NW - 1) / NW;      // (super band, hh) of the band operand per thread
  __shared__ double sA[2][HKR][SA], sB[2][HKR][SB];
  const XcdTile xt = xcd_tile(tr * tb * bands.n, ns);
  if (!xt.valid) return;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, li = lane & 15, lk = lane >> 4, hh = t & 7;
  const int job = xt.inner / (tr * tb), tile = xt.inner - job * tr * tb;
  const int r0 = (tile % tr) * WR, b0 = (tile / tr) * (8 * NC);
  const double2 *__restrict__ psi = bands.psi[job];
  rows.job(job);
  const int h0 = xt.shared * hsplit, h1 = min(nh, h0 + hsplit);
  const int nchunk = (h1 - h0 + HK - 1) / HK;
  dbl4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = dbl4{0.0, 0.0, 0.0, 0.0};
  typename Rows::Row rw;
  rows.init(rw, r0);
  typename Rows::Pre pa;
  Pair pb[NBT];
  size_t off[NBT];
#pragma unroll
  for (int i = 0; i < NBT; ++i) off[i] = (size_t)min(b0 + min((t >> 3) + 8 * NW * i, 8 * NC - 1), nbh - 1) * ngl;
  // index of chunk c for this thread's hh (clamped into the half list)
  auto idx = [&](int c) { return hg[min(h0 + c * HK + hh, nh - 1)]; };
  auto fetch = [&](int c, int2 g) {
    rows.fetch(rw, h0 + c * HK + hh, g, pa);
#pragma unroll
    for (int i = 0; i < NBT; ++i) load_pair(psi, off[i], g, pb[i]);
  };
  auto store = [&](int c, bool self) {
    const int buf = c & 1;
    rows.store(rw, pa, self, h0 + c * HK + hh < h1, sA[buf]);
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
      const int bl = (t >> 3) + 8 * NW * i;
      if (NC % NW != 0 && bl >= 8 * NC) break;
      const Bands2 r = split_pair(pb[i]);
      sB[buf][hh][2 * bl] = r.are;
      sB[buf][hh][2 * bl + 1] = r.bre;
      sB[buf][HK + hh][2 * bl] = r.aim;
      sB[buf][HK + hh][2 * bl + 1] = r.bim;
    }
  };
  int2 g = idx(0);
  fetch(0, g);
  store(0, g.x == g.y);
  g = idx(1);
  for (int c = 0; c < nchunk; ++c) {
    __syncthreads();
    const bool more = c + 1 < nchunk;
    const bool self = g.x == g.y;
    if (more) {
      fetch(c + 1, g);
      g = idx(c + 2);
    }
    const double (*a)[SA] = sA[c & 1];
    const double (*b)[SB] = sB[c & 1];
#pragma unroll
    for (int ks = 0; ks < HKR / 4; ++ks) {
      const int k = 4 * ks + lk;
      const double av = a[k][16 * wv + li];
#pragma unroll
      for (int q = 0; q < NC; ++q) acc[q] = mfma4(av, b[k][16 * q + li], acc[q]);
    }
    if (more) store(c + 1, self);
  }
  double *dst = part + ((size_t)job * ns + xt.shared) * nrow * (2 * nbh);
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int n = 2 * b0 + 16 * q + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = r0 + 16 * wv + lk + 4 * r;
      if (i < nrow && n < 2 * nbh) dst[(size_t)i * (2 * nbh) + n] = acc[q][r];
    }
  }
}

// WAVES_OVERLAP + WAVES_1COVERLAP: the NB x NB matrix from the split partials
// of the real-band product (scaled) and the one-centre runs (c1, c2) of
// k_overlap1c in z order.  One thread per (row n, super band j): two elements;
// blockIdx.y is the matrix.
struct HalfMats {
  double *mat[kOvlJobs];
};
__global__ void __launch_bounds__(kRedC * kRedS) k_half_finish(const double2 *__restrict__ part, int ns, int nb,
                                                               double scale, const double4 *__restrict__ part1c,
                                                               int nz, HalfMats mats) {
  __shared__ double2 red[kRedS][kRedC];
  const int c = threadIdx.x % kRedC, sl = threadIdx.x / kRedC;
  const int nbh = nb / 2, n = nb * nbh, idx = blockIdx.x * kRedC + c;
  part += (size_t)blockIdx.y * ns * n;
  if (part1c) part1c += (size_t)blockIdx.y * nz * nbh * nbh;
  double *mat = mats.mat[blockIdx.y];
  const bool in = idx < n;
  double2 acc = czero();
  if (in) {
    constexpr int V = 8;
    for (int k0 = sl; k0 < ns; k0 += V * kRedS) {
      double2 v[V];
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int k = k0 + u * kRedS;
        v[u] = k < ns ? part[(size_t)k * n + idx] : czero();
      }
#pragma unroll
      for (int u = 0; u < V; ++u) acc = radd(acc, v[u]);
    }
  }
  red[sl][c] = acc;
  __syncthreads();
  if (sl != 0 || !in) return;
  double2 r = red[0][c];
#pragma unroll
  for (int q = 1; q < kRedS; ++q) r = radd(r, red[q][c]);
  r = rscale(r, scale);
  if (part1c) {
    const int row = idx / nbh, j = idx - row * nbh;
    const size_t o = (size_t)(row >> 1) * nbh + j;
    double4 cc = make_double4(0.0, 0.0, 0.0, 0.0);
    for (int z = 0; z < nz; ++z) {
      const double4 v = part1c[(size_t)z * nbh * nbh + o];
      cc.x += v.x;
      cc.y += v.y;
      cc.z += v.z;
      cc.w += v.w;
    }
    if ((row & 1) == 0) {
      r.x += 0.5 * (cc.x + cc.z);
      r.y += 0.5 * (cc.y + cc.w);
    } else {
      r.x += -(0.5 * (cc.y - cc.w));
      r.y += 0.5 * (cc.x - cc.z);
    }
  }
  reinterpret_cast<double2 *>(mat)[idx] = r;
}

// ---------------------------------------------------------------------------
// Column products: psi_b(G) += sum_k x(k, b) B(k, G) for both G of a pair.
// The real products of a real band with the re and im planes of B are kept
// apart, rr = sum x1 re, ir = sum x1 im, ri = sum x2 re, ii = sum x2 im with
// (x1, x2) the coefficients of the two real bands; the pair then gets
//   psi(G) += (rr - ii, ir + ri),  psi(-G) += (rr + ii, ri - ir).
// B: projectors (ADDPRO, x = projections) or the real bands of chi (ADDOPSI,
// x = LAMBDA).
// ---------------------------------------------------------------------------
// (re, im) planes of 16 projectors at 16 G: one (k, h) per thread, t < 256
struct PlaneP {
  HalfP p;
  struct Pre {
    double f;
    double2 e;
    int odd;
  };
  __device__ int4 entry(int k0) const {
    return p.tab[min(k0 + (int)((threadIdx.x & 255) >> 4), p.npro - 1)];
  }
  __device__ void fetch(int4 t, int, int h, int2, Pre &v) const {
    v.odd = t.z;
    if (threadIdx.x >= 256) return;               // whole waves (124 -> 101 us for Si64)
    v.f = p.frow(t)[h];
    v.e = p.erow(t)[h];
  }
  template <int SB>
  __device__ void store(const Pre &v, double (*re)[SB], double (*im)[SB]) const {
    const int t = threadIdx.x;
    if (t >= 256) return;
    const double2 z = rot_odd(make_double2(v.f * v.e.x, v.f * v.e.y), v.odd);
    re[t >> 4][t & 15] = z.x;
    im[t >> 4][t & 15] = z.y;
  }
};

// (re, im) planes of 8 super bands (16 real bands) of chi: t < 128
struct PlaneX {
  const double2 *chi;
  int ngl, nbh;
  struct Pre {
    Pair v;
  };
  __device__ int4 entry(int) const { return make_int4(0, 0, 0, 0); }
  __device__ void fetch(int4, int k0, int, int2 g, Pre &p) const {
    const int b = k0 / 2 + ((threadIdx.x & 127) >> 4);
    load_pair(chi, (size_t)min(b, nbh - 1) * ngl, g, p.v);
  }
  template <int SB>
  __device__ void store(const Pre &p, double (*re)[SB], double (*im)[SB]) const {
    const int t = threadIdx.x, k = 2 * (t >> 4), h = t & 15;
    if (t >= 128) return;
    // the real bands c = half the sums
    const Bands2 r = split_pair(p.v);
    re[k][h] = 0.5 * r.are;
    re[k + 1][h] = 0.5 * r.bre;
    im[k][h] = 0.5 * r.aim;
    im[k + 1][h] = 0.5 * r.bim;
  }
};

// Workgroup: 16 G pairs x nt tiles of 8 super bands; wave w < nt / RTW takes
// tiles w RTW .. with two accumulators each (at least four waves, so that 256
// threads stage B).  One tile per wave keeps many small waves per CU and one
// G block per workgroup keeps the last wave of workgroups full (746 blocks
// at Si64); the coefficients, 8 NPRO NB bytes per workgroup, come from L2.
// Row i of a tile's MFMA is real band 2 b + part with i = (b & 3) | part << 2 |
// (b >> 2) << 3, so a lane's four results are (c1, c2) of two super bands.
template <class Plane, int RTW>
__global__ void __launch_bounds__(1024) k_half_col(Plane pl, const double2 *__restrict__ x,
                                                   const int2 *__restrict__ hg, int nk, int nh, int ngl, int nbh,
                                                   int nt, ColOut out) {
  extern __shared__ double sm[];
  constexpr int SB = hpad(16);
  const int SA = hpad(16 * nt);
  double (*sRe)[SB] = reinterpret_cast<double (*)[SB]>(sm);            // [2][16][SB]
  double (*sIm)[SB] = sRe + 2 * 16;
  double *sA = sm + 4 * 16 * SB;                                      // [2][16][SA]
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, li = lane & 15, lk = lane >> 4;
  const int h0 = blockIdx.x * 16, b0 = blockIdx.y * 8 * nt, nw = 8 * nt;
  const int hs = h0 + (t & 15);
  const int2 g = hg[min(hs, nh - 1)];
  // this thread's coefficients: element e = t + i blockDim of the chunk's 16 x nw
  constexpr int NA = 2 * RTW;
  // (those of rows beyond nk are zero, those of bands beyond nbh go unused),
  // its place in the row and in LDS
  int ka[NA], da[NA], oa[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int e = t + i * blockDim.x;
    ka[i] = e / nw;
    const int bl = e - ka[i] * nw;
    oa[i] = (ka[i] & 15) * nbh + min(b0 + bl, nbh - 1);
    da[i] = ka[i] * SA + 16 * (bl >> 3) + (bl & 3) + ((bl >> 2) & 1) * 8;
  }
  double2 va[NA];
  typename Plane::Pre pre;
  auto fetch = [&](int k0, int4 ent) {
    pl.fetch(ent, k0, hs, g, pre);
    const double2 *xc = x + (size_t)k0 * nbh;
#pragma unroll
    for (int i = 0; i < NA; ++i) va[i] = k0 + ka[i] < nk ? xc[oa[i]] : czero();
  };
  auto store = [&](int buf) {
    pl.store(pre, sRe + 16 * buf, sIm + 16 * buf);
    double *d = sA + buf * 16 * SA;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      if (ka[i] >= 16) continue;
      d[da[i]] = va[i].x;
      d[da[i] + 4] = va[i].y;
    }
  };
  dbl4 ar[RTW], ai[RTW];
#pragma unroll
  for (int r = 0; r < RTW; ++r) {
    ar[r] = dbl4{0.0, 0.0, 0.0, 0.0};
    ai[r] = dbl4{0.0, 0.0, 0.0, 0.0};
  }
  const bool on = wv * RTW < nt;
  int4 ent = pl.entry(0);
  fetch(0, ent);
  ent = pl.entry(16);
  store(0);
  const int nchunk = (nk + 15) / 16;
  for (int c = 0; c < nchunk; ++c) {
    __syncthreads();
    const bool more = c + 1 < nchunk;
    if (more) {
      fetch(16 * (c + 1), ent);
      ent = pl.entry(16 * (c + 2));
    }
    if (on) {
      const int buf = 16 * (c & 1);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int k = buf + 4 * ks + lk;
        const double br = sRe[k][li], bi = sIm[k][li];
#pragma unroll
        for (int r = 0; r < RTW; ++r) {
          const double av = sA[(size_t)k * SA + 16 * min(wv * RTW + r, nt - 1) + li];
          ar[r] = mfma4(av, br, ar[r]);
          ai[r] = mfma4(av, bi, ai[r]);
        }
      }
    }
    if (more) store((c + 1) & 1);
  }
  const int h = h0 + li;
  if (!on || h >= nh) return;
  const int2 gg = hg[h];
#pragma unroll
  for (int r = 0; r < RTW; ++r) {
    const int tile = wv * RTW + r;
    if (tile >= nt) break;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int b = b0 + 8 * tile + 4 * q + lk;
      if (b >= nbh) continue;
      const double rr = ar[r][2 * q], ri = ar[r][2 * q + 1], ir = ai[r][2 * q], ii = ai[r][2 * q + 1];
      const size_t o = (size_t)b * ngl;
      out.store(o + gg.x, gg.x, rr - ii, ir + ri);
      if (gg.x != gg.y) out.store(o + gg.y, gg.y, rr + ii, ri - ir);
    }
  }
}

// ---------------------------------------------------------------------------
// Forces (WAVES_DEDPRO + WAVES_PROFORCE): D'(i,h) = sum_n ded(i,n) X(n,h) over
// the real bands is twice the INVERTG-symmetrised dE/dP; with P(-G) =
// conj(P(G)) the terms of G and -G are equal, so
// F(i) = 2 Omega sum_h G Re[i P conj(D')].  part[htile][i][3] sums 32 G pairs.
// Workgroup: four waves, 32 projector rows each, two blocks of 16 G pairs;
// the real-band planes of a chunk are staged once for 128 rows.
// ---------------------------------------------------------------------------
constexpr int kFW = 4, kFRT = 2, kFHT = 2;
__global__ void __launch_bounds__(64 * kFW, 2) k_half_force(HalfP p, const double2 *__restrict__ ded,
                                                            const double2 *__restrict__ psi,
                                                            const int2 *__restrict__ hg, int nh, int ngl, int nbh,
                                                            const double *__restrict__ gvec, int nrt, int nht,
                                                            double *__restrict__ part) {
  constexpr int WR = 16 * kFW * kFRT, SA = hpad(WR), WH = 16 * kFHT, SB = hpad(WH);
  __shared__ double sA[2][16][SA], sRe[2][16][SB], sIm[2][16][SB];
  const XcdTile xt = xcd_tile(nrt, nht);
  if (!xt.valid) return;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, li = lane & 15, lk = lane >> 4;
  const int r0 = xt.inner * WR, h0 = xt.shared * WH;
  const int hb = t & (WH - 1), bb = t / WH;               // band operand: (pair, super band of the chunk)
  const int2 g = hg[min(h0 + hb, nh - 1)];              // (the columns beyond NH and the term G = 0 get no weight)
  constexpr int NA = WR * 8 / (64 * kFW);
  const int ba = t & 7;
  const double2 *da[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) da[i] = ded + (size_t)min(r0 + (t >> 3) + 8 * kFW * i, p.npro - 1) * nbh;
  double2 va[NA];
  Pair pb;
  auto fetch = [&](int c) {
    load_pair(psi, (size_t)min(8 * c + bb, nbh - 1) * ngl, g, pb);
    const int bk = 8 * c + ba, bc = min(bk, nbh - 1);
#pragma unroll
    for (int i = 0; i < NA; ++i) va[i] = da[i][bc];
    if (bk >= nbh) {                                      // rows of the contraction beyond the bands
#pragma unroll
      for (int i = 0; i < NA; ++i) va[i] = czero();
    }
  };
  auto store = [&](int buf) {
    const Bands2 x = split_pair(pb);
    sRe[buf][2 * bb][hb] = x.are;
    sRe[buf][2 * bb + 1][hb] = x.bre;
    sIm[buf][2 * bb][hb] = x.aim;
    sIm[buf][2 * bb + 1][hb] = x.bim;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int r = (t >> 3) + 8 * kFW * i;
      sA[buf][2 * ba][r] = va[i].x;
      sA[buf][2 * ba + 1][r] = va[i].y;
    }
  };
  dbl4 ar[kFRT][kFHT], ai[kFRT][kFHT];
#pragma unroll
  for (int r = 0; r < kFRT; ++r)
#pragma unroll
    for (int q = 0; q < kFHT; ++q) {
      ar[r][q] = dbl4{0.0, 0.0, 0.0, 0.0};
      ai[r][q] = dbl4{0.0, 0.0, 0.0, 0.0};
    }
  fetch(0);
  store(0);
  const int nchunk = (nbh + 7) / 8;
  for (int c = 0; c < nchunk; ++c) {
    __syncthreads();
    const bool more = c + 1 < nchunk;
    if (more) fetch(c + 1);
    const int buf = c & 1;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int k = 4 * ks + lk;
      double br[kFHT], bi[kFHT];
#pragma unroll
      for (int q = 0; q < kFHT; ++q) {
        br[q] = sRe[buf][k][16 * q + li];
        bi[q] = sIm[buf][k][16 * q + li];
      }
#pragma unroll
      for (int r = 0; r < kFRT; ++r) {
        const double av = sA[buf][k][16 * (wv * kFRT + r) + li];
#pragma unroll
        for (int q = 0; q < kFHT; ++q) {
          ar[r][q] = mfma4(av, br[q], ar[r][q]);
          ai[r][q] = mfma4(av, bi[q], ai[r][q]);
        }
      }
    }
    if (more) store((c + 1) & 1);
  }
  double gx[kFHT], gy[kFHT], gz[kFHT];
#pragma unroll
  for (int q = 0; q < kFHT; ++q) {
    const int h = h0 + 16 * q + li, ig = h < nh ? hg[h].x : 0;
    gx[q] = h < nh ? gvec[3 * ig] : 0.0;
    gy[q] = h < nh ? gvec[3 * ig + 1] : 0.0;
    gz[q] = h < nh ? gvec[3 * ig + 2] : 0.0;
  }
#pragma unroll
  for (int rt = 0; rt < kFRT; ++rt) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ip = r0 + 16 * (wv * kFRT + rt) + lk + 4 * r;
      double f[3] = {0.0, 0.0, 0.0};
      if (ip < p.npro) {
        const int4 tb = p.tab[ip];
#pragma unroll
        for (int q = 0; q < kFHT; ++q) {
          const int h = h0 + 16 * q + li;                 // < NHP: zero tables beyond NH
          const double s = p.frow(tb)[h];
          const double2 e = p.erow(tb)[h];
          const double2 pv = rot_odd(make_double2(s * e.x, s * e.y), tb.z);
          // Re(i p conj(d)) = p.x d.y - p.y d.x
          const double cc = pv.x * ai[rt][q][r] - pv.y * ar[rt][q][r];
          f[0] += cc * gx[q];
          f[1] += cc * gy[q];
          f[2] += cc * gz[q];
        }
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) f[d] = row16_sum(f[d]);
      if (li == 0 && ip < p.npro) {
        double *dst = part + ((size_t)xt.shared * p.npro + ip) * 3;
        dst[0] = f[0];
        dst[1] = f[1];
        dst[2] = f[2];
      }
    }
  }
}

constexpr int kHalfMinChunks = 2;   // K chunks per G split of a row product at least

// part[split][nrow][2 nbh] = rows x bands; the split count follows the
// autotuned number of waves (about two per SIMD by default)
template <int NW, class Rows>
int run_half_row(pw_waveset *ws, const Rows &rows, int nrow, const HalfBands &bands, int *ns_out, const char *name) {
  pw_plan *p = ws->plan;
  const int nbh = ws->nbh, nh = p->nh;
  const int ct = (2 * nbh + 15) / 16;              // blocks of 16 real bands, at most 9 per workgroup
  const int tb = (ct + 8) / 9, nc = (ct + tb - 1) / tb;
  const int tr = (nrow + 16 * NW - 1) / (16 * NW);
  const int chunks = (nh + HK - 1) / HK;
  const int want = std::max(1, ws->tune_split_waves / NW / std::max(1, tr * tb * bands.n));
  int ns = std::max(1, std::min(want, chunks / kHalfMinChunks));
  const int hsplit = (chunks + ns - 1) / ns * HK;
  ns = (nh + hsplit - 1) / hsplit;
  PW_TRY(ws_part(ws, (size_t)bands.n * ns * nrow * 2 * nbh * sizeof(double)));
  {
    ScopeTimer tm(ws, name);
    const unsigned grid = xcd_blocks(tr * tb * bands.n, ns);
#define PW_LAUNCH(NC)                                                                                       \
  case NC:                                                                                                  \
    k_half_row<Rows, NC, NW><<<grid, 64 * NW, 0, ws->stream>>>(rows, bands, p->d_hg, nh, nrow, p->ngl, nbh,   \
                                                               hsplit, tr, tb, ns, ws->d_part);             \
    break;
    switch (nc) {
      PW_LAUNCH(1) PW_LAUNCH(2) PW_LAUNCH(3) PW_LAUNCH(4) PW_LAUNCH(5) PW_LAUNCH(6) PW_LAUNCH(7) PW_LAUNCH(8)
      PW_LAUNCH(9)
    }
#undef PW_LAUNCH
    PW_HIP(hipGetLastError());
  }
  *ns_out = ns;
  return PW_OK;
}

// psi += x B over tiles of 8 super bands: up to 16 tiles one per wave, more two per wave, at most 32 per workgroup
template <class Plane>
int run_half_col(pw_waveset *ws, const Plane &pl, const double2 *x, int nk, const ColOut &out, const char *name) {
  pw_plan *p = ws->plan;
  const int nbh = ws->nbh, rt = (nbh + 7) / 8;
  const int grp = (rt + 31) / 32, nt = (rt + grp - 1) / grp, rtw = nt > 16 ? 2 : 1;
  const int nw = std::max(4, (nt + rtw - 1) / rtw);
  const size_t lds = (size_t)(4 * 16 * hpad(16) + 2 * 16 * hpad(16 * nt)) * sizeof(double);
  const dim3 grid((p->nh + 15) / 16, grp);
  ScopeTimer tm(ws, name);
  auto fn = rtw == 1 ? k_half_col<Plane, 1> : k_half_col<Plane, 2>;
  if (lds > 65536) {
    // the 160 KiB of a CU (nt <= 32 takes 141 KiB), once per process
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
      for (const void *f : {(const void *)k_half_col<Plane, 1>, (const void *)k_half_col<Plane, 2>}) {
        const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) err = e;
      }
    });
    PW_HIP(err);
  }
  fn<<<grid, 64 * nw, lds, ws->stream>>>(pl, x, p->d_hg, nk, p->nh, p->ngl, nbh, nt, out);
  PW_HIP(hipGetLastError());
  return PW_OK;
}

HalfP half_p(const pw_waveset *ws) {
  const int nhp = half_pad(ws->plan);
  const double *f = (const double *)ws->d_hfac;
  return HalfP{f, (const double2 *)(f + (size_t)ws->nsp * ws->lmnxx * nhp), ws->d_ipro4, ws->npro, nhp};
}

}  // namespace

// device room of the projector factors on the half list: [F][E], NHP is a
// multiple of 32, so E starts 16-byte aligned
int half_factors_room(pw_waveset *ws) {
  const size_t nhp = half_pad(ws->plan);
  const size_t bytes = nhp * ((size_t)ws->nsp * ws->lmnxx * sizeof(double) + ws->nat * sizeof(double2));
  if (bytes <= ws->hfac_bytes) return PW_OK;
  if (ws->d_hfac) PW_HIP(hipFree(ws->d_hfac));
  ws->d_hfac = nullptr;
  ws->hfac_bytes = 0;
  PW_HIP(hipMalloc(&ws->d_hfac, bytes));
  ws->hfac_bytes = bytes;
  return PW_OK;
}

// projector factors on the half list for the positions of the phase tables
int half_factors(pw_waveset *ws) {
  pw_plan *p = ws->plan;
  const int nhp = half_pad(p);
  const size_t nf = (size_t)ws->nsp * ws->lmnxx * nhp, ne = (size_t)ws->nat * nhp;
  PW_TRY(half_factors_room(ws));   // a mixed set that evaluates ORTHOERR has none yet
  ProjGeo q = make_pgeo(ws);
  double *f = (double *)ws->d_hfac;
  ScopeTimer tm(ws, "pgen");
  k_half_f<<<(nf + 255) / 256, 256, 0, ws->stream>>>(q, ws->nsp, p->nh, nhp, p->d_hg, f);
  k_half_e<<<(ne + 255) / 256, 256, 0, ws->stream>>>(q, p->nh, nhp, p->d_hg, (double2 *)(f + nf));
  PW_HIP(hipGetLastError());
  return PW_OK;
}

int half_projections(pw_waveset *ws, const double2 *psi, double2 *proj) {
  RowsP<4> rows{half_p(ws)};
  int ns = 0;
  PW_TRY(run_half_row<4>(ws, rows, ws->npro, HalfBands{{psi}, 1}, &ns, "projections"));
  const size_t n = (size_t)ws->npro * ws->nbh;
  ScopeTimer tm(ws, "reduce");
  k_reduce_split<double2><<<(n + kRedC - 1) / kRedC, kRedC * kRedS, 0, ws->stream>>>((const double2 *)ws->d_part, ns,
                                                                                       (int)n, ws->plan->vol, proj);
  PW_HIP(hipGetLastError());
  return PW_OK;
}

// mat = Omega sum conj(c_i) c_j (+ the one-centre runs p1c) for the matrices of
// jobs; a workgroup of three waves when that wastes fewer 16-row blocks than
// four.  One launch each for all matrices: they share the reads of the wave
// functions in an XCD's L2, and a small set's are bound by launches.  The three
// of a CP step: Si8 13.4 + 9.4 (finishing passes) -> 5.3 + 3.7 us, Si64 (144
// bands) 108 -> 82 and one finishing pass of 9.8.
int half_overlap(pw_waveset *ws, const OverlapJob *jobs, int nj, const double4 *p1c, int nz) {
  const int nb = 2 * ws->nbh, mt = (nb + 15) / 16;
  HalfBands bands{};
  HalfMats mats{};
  bands.n = nj;
  for (int j = 0; j < nj; ++j) {
    bands.psi[j] = jobs[j].psi2;
    mats.mat[j] = jobs[j].mat;
  }
  auto rows = [&](auto r) {
    for (int j = 0; j < nj; ++j) r.psis[j] = jobs[j].psi1;
    r.ngl = ws->plan->ngl;
    r.nbh = ws->nbh;
    return r;
  };
  int ns = 0;
  if ((mt + 2) / 3 * 3 < (mt + 3) / 4 * 4) PW_TRY(run_half_row<3>(ws, rows(RowsX<3>{}), nb, bands, &ns, "overlap"));
  else PW_TRY(run_half_row<4>(ws, rows(RowsX<4>{}), nb, bands, &ns, "overlap"));
  ScopeTimer tm(ws, "reduce");
  const int n = nb * ws->nbh;
  k_half_finish<<<dim3((n + kRedC - 1) / kRedC, nj), kRedC * kRedS, 0, ws->stream>>>(
      (const double2 *)ws->d_part, ns, nb, 0.5 * ws->plan->vol, p1c, nz, mats);
  PW_HIP(hipGetLastError());
  return PW_OK;
}

int half_addpro(pw_waveset *ws, const ColOut &out, const double2 *x) {
  PlaneP pl{half_p(ws)};
  return run_half_col(ws, pl, x, ws->npro, out, "addpro");
}

// psibar_j += sum_i chi_i LAMBDA(i,j) over the real bands; LAMBDA is row-major
// NB x NB, so row i is NBH pairs (LAMBDA(i,2b), LAMBDA(i,2b+1))
int half_addopsi(pw_waveset *ws, double2 *psibar, const double2 *chi, const double *lam) {
  PlaneX pl{chi, ws->plan->ngl, ws->nbh};
  return run_half_col(ws, pl, (const double2 *)lam, ws->nb, ColOut{psibar, nullptr, nullptr, 0.0}, "addopsi");
}

int half_force(pw_waveset *ws, const double2 *psi, const double2 *ded, double *dst) {
  pw_plan *p = ws->plan;
  const int nht = (p->nh + 16 * kFHT - 1) / (16 * kFHT), nrt = (ws->npro + 16 * kFW * kFRT - 1) / (16 * kFW * kFRT);
  const size_t n = (size_t)ws->npro * 3;
  PW_TRY(ws_part(ws, (size_t)nht * n * sizeof(double)));
  {
    ScopeTimer tm(ws, "force");
    k_half_force<<<xcd_blocks(nrt, nht), 64 * kFW, 0, ws->stream>>>(half_p(ws), ded, psi, p->d_hg, p->nh, p->ngl,
                                                                    ws->nbh, p->d_gvec, nrt, nht, ws->d_part);
    PW_HIP(hipGetLastError());
  }
  k_reduce_split<double><<<(n + kRedC - 1) / kRedC, kRedC * kRedS, 0, ws->stream>>>(ws->d_part, nht, (int)n,
                                                                                      2.0 * p->vol, dst);
  PW_HIP(hipGetLastError());
  return PW_OK;
}
