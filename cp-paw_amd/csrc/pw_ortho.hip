// WAVES_ORTHO_X (src/paw_waves2.f90:1844-2022) in FP64 on the GPU.
//
// The reference iterates
//   GAMN   = sym[LAMBDA^T (CHICHI LAMBDA + 2 CHIPSI)] + PSIPSI - 1
//   LAMBDA -= 2 f_i/(f_i+f_j) * S^-1(GAMN),   S(X) = B X + X B,  B = sym(CHIPSI)
// until max|GAMN| < 1e-8, applying S^-1 through the eigenvectors of B (DSYEV).
// The iterates depend on S^-1 only, not on an eigen-basis, so this
// implementation keeps the reference's outer iteration and stopping rule and
// applies S^-1 exactly (to rounding) with GEMMs only, as a series from the
// Cayley transform:
//   M = (B + qI)^-1 (Newton-Schulz), A = I - 2qM = (B - qI)M,
//   S^-1(G) = 2q sum_{k<K} P_k G P_k,  P_k = A^k M (symmetric), K = 2^J;
//   the error after K terms is rho^(2K), rho = (sqrt(k)-1)/(sqrt(k)+1) for
//   the spectral bounds of B (Lanczos on the device, widened).  B is
//   positive definite in the CP step (B ~ dt^2/m); for a B that is not
//   (or too ill-conditioned for the series) S^-1 is applied as the reference
//   does, through the eigenvectors of B, which one workgroup computes by
//   cyclic Jacobi rotations (ortho_x_eig).  The P_k are formed once
//   per call (up to 8 in one launch, more by doubling, one row-panel batch
//   launch per level); each outer
//   iteration then applies the series in two launches (row-panel chains
//   P_k G P_k, then the ordered sum over k with the convergence test and the
//   LAMBDA update).  Only terms beyond 2^5 would continue by the Smith
//   recursion X <- X + A_j X A_j, A_j = A^(2^j); no tested cell needs them.
// On the series path every product is an NB^3 FP64-MFMA GEMM and nothing is
// diagonalised.  The
// outer loop runs on the device: the convergence test sets a flag that makes
// every later kernel of the batch return at once, so the host waits only
// once per batch of iterations (batch = the previous call's count).  Sets
// whose matrices fit in LDS are solved by one workgroup in one launch.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "pw_common.h"
#include "pw_device.h"

namespace {

typedef double dbl2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int T16 = 16;
constexpr int kMaxLevels = 12;
constexpr int kMaxIter = 200;      // src/paw_waves2.f90:1870 (NITERX)
constexpr int kLzThreads = 1024;
constexpr int kLzMaxSteps = 30;

// Loop state of one ORTHO_X call, written by the convergence test in each
// iteration's k_series_sum (the first one also applies the acceptance test of
// the preparation) and reset by k_ns_first.
struct OrthoState {
  int done;   // 1 once converged or failed
  int iter;   // iteration at which max|GAMN| < tolerance
  int code;   // 0 ok, 1 NaN, 2 divergence
  int passes; // passes over the terms of the series (iterations that form S^-1(GAMN))
};

__device__ inline bool stopped(const OrthoState *st) { return st != nullptr && st->done != 0; }

// C = alpha op(A) op(B) + beta D   (row-major n x n) on FP64 MFMA.
// One 16x16 tile of C per workgroup; its eight waves take interleaved K slices
// of four (all loads of a wave issued before its MFMAs, one memory round trip
// for n <= 256) and are summed through LDS in a fixed order.  Lane layout of
// v_mfma_f64_16x16x4f64: A(i,k) in lane i+16k, B(k,j) in lane j+16k, C(i,j)
// in lane j+16(i%4), element i/4.
constexpr int kGemmWaves = 8;
__device__ __forceinline__ void gemm_tile(int n, const double *__restrict__ A, int ta,
                                          const double *__restrict__ B, int tb, double *C, double alpha,
                                          const double *D, double beta, int i0, int j0,
                                          dbl4 (*part)[64]) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int ia = i0 + li, jb = j0 + li;
  const bool aok = ia < n, bok = jb < n;
  dbl4 acc = {0.0, 0.0, 0.0, 0.0};
  const int nk = (n + 3) / 4;
  constexpr int U = 8;
  for (int ks0 = wv; ks0 < nk; ks0 += kGemmWaves * U) {
    double a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 4 * (ks0 + kGemmWaves * u) + lk;
      a[u] = 0.0;
      b[u] = 0.0;
      if (k < n) {
        if (aok) a[u] = ta ? A[(size_t)k * n + ia] : A[(size_t)ia * n + k];
        if (bok) b[u] = tb ? B[(size_t)jb * n + k] : B[(size_t)k * n + jb];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc, 0, 0, 0);
  }
  if (wv > 0) part[wv - 1][lane] = acc;
  __syncthreads();
  if (wv != 0) return;
#pragma unroll
  for (int w = 0; w < kGemmWaves - 1; ++w) acc += part[w][lane];
  const int j = j0 + li;
  if (j >= n) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + lk + 4 * r;
    if (i < n) {
      double v = alpha * acc[r];
      if (D) v += beta * D[(size_t)i * n + j];
      C[(size_t)i * n + j] = v;
    }
  }
}

__global__ void __launch_bounds__(64 * kGemmWaves) k_gemm(int n, const double *__restrict__ A, int ta,
                                                          const double *__restrict__ B, int tb, double *C,
                                                          double alpha, const double *D, double beta,
                                                          const OrthoState *st) {
  if (stopped(st)) return;
  __shared__ dbl4 part[kGemmWaves - 1][64];
  gemm_tile(n, A, ta, B, tb, C, alpha, D, beta, blockIdx.y * T16, blockIdx.x * T16, part);
}

// Row panels.  A workgroup of kPanelWaves waves forms a 16 x n row panel of
// an n x n product: the A row panel is staged in LDS once and the waves take
// the 16 x 16 column tiles j = w, w + kPanelWaves, ... each over the whole K
// (no split of K, no reduction).  The B operand of a tile is loaded in
// chunks of kKC MFMA steps, all loads of a chunk issued before its MFMAs:
// one memory round trip per tile for n <= 4 kKC.  B is row-major n x n,
// TB = 0: B(k, j) = B[k n + j], TB = 1: B(k, j) = B[j n + k].
constexpr int kPanelWaves = 9;   // one wave per column tile at NB = 144
constexpr int kKC = 36;

// B operand of one chunk: b[u] = B(4 (s0 + u) + lk, j0 + li).  Row and
// column indices are clamped into the matrix, so every load is valid and
// unpredicated; a clamped row k >= n meets a zero A column (the LDS pad) and
// a clamped column j >= n gives an output column that is not stored.
template <int TB>
__device__ __forceinline__ void load_bchunk(double (&b)[kKC], int n, const double *__restrict__ B, int j0,
                                            int s0) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int jc = min(j0 + li, n - 1);
#pragma unroll
  for (int u = 0; u < kKC; ++u) {
    const int kc = min(4 * (s0 + u) + lk, n - 1);
    b[u] = TB ? B[(size_t)jc * n + kc] : B[(size_t)kc * n + jc];
  }
}

// acc += A(:, chunk) B(chunk, tile), A(i, k) = sA[i ldr + k] in LDS; columns
// n..ldr-1 of sA are zero and k is clamped to them
__device__ __forceinline__ void mfma_chunk(dbl4 &acc, const double (&b)[kKC], const double *sA, int ldr, int s0) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int u = 0; u < kKC; ++u) {
    const double av = sA[li * ldr + min(4 * (s0 + u) + lk, ldr - 1)];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[u], acc, 0, 0, 0);
  }
}

// the chunks s0 >= s1 of one tile (the earlier ones come prefetched)
template <int TB>
__device__ __forceinline__ void panel_rest(dbl4 &acc, int n, const double *sA, int ldr,
                                           const double *__restrict__ B, int j0, int s1) {
  const int nk = (n + 3) / 4;
#pragma unroll 1
  for (int s0 = s1; s0 < nk; s0 += kKC) {
    double b[kKC];
    load_bchunk<TB>(b, n, B, j0, s0);
    mfma_chunk(acc, b, sA, ldr, s0);
  }
}

// A rows 0..15 of a row panel (rows >= nr zero) into sA[16][ldr], columns
// n..ldr-1 zero
__device__ __forceinline__ void stage_panel(int n, const double *__restrict__ A, int nr, double *sA, int ldr) {
  for (int e = threadIdx.x; e < T16 * ldr; e += blockDim.x) {
    const int i = e / ldr, k = e - i * ldr;
    sA[e] = (i < nr && k < n) ? A[(size_t)i * n + k] : 0.0;
  }
}

// LDS row stride of a staged panel: >= n + 1 (a zero pad column) and == 2
// (mod 32) doubles, so the 32 lanes of a half-wave reading A(li, 4s + lk)
// hit distinct bank pairs
__host__ __device__ inline int panel_ldr(int n) { return n + 1 + ((1 - n) % 32 + 32) % 32; }

constexpr size_t kLdsMax = 160 * 1024;
inline size_t panel_lds(int n) { return (size_t)T16 * panel_ldr(n) * sizeof(double); }
// the terms of the series side by side where their launch is bound by latency
// and occupancy, up to the sets whose two 16-row panels fit in LDS; wider ones
// take the Smith levels, half the products
inline bool series_fits(int n) { return 2 * panel_lds(n) + 1024 <= kLdsMax; }

// Batched products with one shared left operand, by row panels:
//   C_z = A B_z,  B_z = B + z sb, C_z = C + z sc,  z < nz,
// and, when Bx is set, one more member z = nz: Cx = A Bx.
// Grid (row panel, member).
struct BatchArgs {
  int n, nz;
  const double *A;
  const double *B;
  size_t sb;
  double *C;
  size_t sc;
  const double *Bx;
  double *Cx;
};

__global__ void __launch_bounds__(64 * kPanelWaves) k_panel_batch(BatchArgs a) {
  extern __shared__ double sA[];   // 16 x ldr
  const int n = a.n, nt = (n + T16 - 1) / T16, ldr = panel_ldr(n);
  const int z = blockIdx.y, I0 = blockIdx.x * T16;
  const double *B = z < a.nz ? a.B + (size_t)z * a.sb : a.Bx;
  double *C = z < a.nz ? a.C + (size_t)z * a.sc : a.Cx;
  const int wv = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  double b0[kKC];
  if (wv < nt) load_bchunk<0>(b0, n, B, wv * T16, 0);
  stage_panel(n, a.A + (size_t)I0 * n, n - I0, sA, ldr);
  __syncthreads();
#pragma unroll 1
  for (int jt = wv; jt < nt; jt += kPanelWaves) {
    dbl4 acc = {0.0, 0.0, 0.0, 0.0};
    if (jt == wv) {
      mfma_chunk(acc, b0, sA, ldr, 0);
      panel_rest<0>(acc, n, sA, ldr, B, jt * T16, kKC);
    } else {
      panel_rest<0>(acc, n, sA, ldr, B, jt * T16, 0);
    }
    const int j = jt * T16 + li;
    if (j >= n) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = I0 + lk + 4 * r;
      if (i < n) C[(size_t)i * n + j] = acc[r];
    }
  }
}

// Tile pairs.  k_gemm_pair computes the tile (I,J) of
// C = alpha op(A) op(B) + beta D and also the tile (J,I), both with the same
// K slicing and summation order as k_gemm (so every element has the value
// k_gemm gives it), and finishes in the epilogue an elementwise step that
// needs C(i,j) and C(j,i), which saves a launch:
//   kPairGamma:   GAMN(i,j) = 0.5 (C(i,j) + C(j,i)) + PSIPSI(min,max) - delta
//                 and the block maxima of |GAMN|;
//   kPairLambda:  the LAMBDA update (src/paw_waves2.f90:1979-2005) with X = C:
//                   L'(i,j) = L(i,j) - 2 (f_i+ds)/(f_i+f_j+2ds) X(i,j)
//                   Lnew(i,j) = L'(j,i) (f_i+ds)/(f_j+ds) if f_i < f_j, else L'(i,j)
constexpr int kPairGamma = 0, kPairLambda = 1;

struct PairArgs {
  int n;
  const double *A, *B, *D;
  int ta, tb;
  double alpha, beta;
  double *out;                   // GAMN or the new LAMBDA
  const double *psipsi;          // kPairGamma
  double *bmax;                  // kPairGamma: per-workgroup max |GAMN|
  const double *occ, *lam;       // kPairLambda
};

__device__ inline double nanmax2(double a, double b) { return (a != a) ? a : ((b != b) ? b : fmax(a, b)); }
__device__ inline double nanmax(double a, double b) { return (a != a || b != b) ? NAN : fmax(a, b); }

template <int MODE>
__global__ void __launch_bounds__(64 * kGemmWaves) k_gemm_pair(PairArgs a, OrthoState *st) {
  if (stopped(st)) return;
  __shared__ dbl4 part[2][kGemmWaves - 1][64];
  __shared__ double sT[16][17];
  const int n = a.n;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int I0 = blockIdx.y * T16, J0 = blockIdx.x * T16;
  const int nk = (n + 3) / 4;
  constexpr int U = 8;
  dbl4 acc[2] = {dbl4{0.0, 0.0, 0.0, 0.0}, dbl4{0.0, 0.0, 0.0, 0.0}};
  // rows/columns of tile 0 = (I,J) and tile 1 = (J,I); the loads of both
  // tiles are issued together (one memory round trip for n <= 256)
  const int ia0 = I0 + li, jb0 = J0 + li, ia1 = J0 + li, jb1 = I0 + li;
  for (int ks0 = wv; ks0 < nk; ks0 += kGemmWaves * U) {
    double av[2][U], bv[2][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 4 * (ks0 + kGemmWaves * u) + lk;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int ia = h == 0 ? ia0 : ia1, jb = h == 0 ? jb0 : jb1;
        av[h][u] = 0.0;
        bv[h][u] = 0.0;
        if (k < n) {
          if (ia < n) av[h][u] = a.ta ? a.A[(size_t)k * n + ia] : a.A[(size_t)ia * n + k];
          if (jb < n) bv[h][u] = a.tb ? a.B[(size_t)jb * n + k] : a.B[(size_t)k * n + jb];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[h][u], bv[h][u], acc[h], 0, 0, 0);
  }
  if (wv > 0) {
    part[0][wv - 1][lane] = acc[0];
    part[1][wv - 1][lane] = acc[1];
  }
  __syncthreads();
  double cv[4];
  if (wv == 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int w = 0; w < kGemmWaves - 1; ++w) acc[h] += part[h][w][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // element (i, j) of tile h: rows of the tile's first index
        const int i = (h == 0 ? I0 : J0) + lk + 4 * r, j = (h == 0 ? J0 : I0) + li;
        double v = a.alpha * acc[h][r];
        if (a.D && i < n && j < n) v += a.beta * a.D[(size_t)i * n + j];
        if (h == 0) cv[r] = v;
        else sT[lk + 4 * r][li] = v;      // C(J+jj, I+ii) at sT[jj][ii]
      }
    }
  }
  __syncthreads();
  double bmx = 0.0;
  if (wv == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ti = lk + 4 * r, i = I0 + ti, j = J0 + li;
      if (i >= n || j >= n) continue;
      const double cij = cv[r], cji = sT[li][ti];
      if (MODE == kPairGamma) {
        const int lo = min(i, j), hi = max(i, j);
        double v = 0.5 * (cij + cji) + a.psipsi[(size_t)lo * n + hi];
        if (i == j) v -= 1.0;
        a.out[(size_t)i * n + j] = v;
        bmx = nanmax2(bmx, (v != v) ? v : fabs(v));
      } else {
        const double oi = a.occ[i] + 1.0e-12, oj = a.occ[j] + 1.0e-12;
        if (a.occ[i] < a.occ[j]) {
          const double lt = a.lam[(size_t)j * n + i] - 2.0 * oj / (oj + oi) * cji;
          a.out[(size_t)i * n + j] = lt * oi / oj;
        } else {
          a.out[(size_t)i * n + j] = a.lam[(size_t)i * n + j] - 2.0 * oi / (oi + oj) * cij;
        }
      }
    }
  }
  if (MODE != kPairGamma) return;
  // block maximum of |GAMN| (NaN propagates); the next kernel of the
  // iteration (k_series_sum) applies the convergence test
  if (wv == 0) {
    double m = bmx;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = nanmax2(m, __shfl_xor(m, o));
    if (lane == 0) a.bmax[blockIdx.y * gridDim.x + blockIdx.x] = m;
  }
}

// The Smith sum written out as a series (the Cayley series of S^-1):
//   S^-1(G) = 2q sum_{k<K} A^k M G M A^k = 2q sum_k P_k G P_k^T,  P_k = A^k M,
// with the P_k formed once per call.  k_series_terms: workgroup (row panel
// I, term k) forms R = P_k(I,:) G into LDS and then the row panel
// part_k(I,:) = R P_k (P_k is symmetric), so each term is a chain of two
// row-panel products inside one workgroup.  k_series_sum adds the K terms of each element in
// the order k = 0, 1, ..., and finishes with
//   kSeriesX:      out = scale * sum            (Smith levels follow), or
//   kSeriesLambda: the LAMBDA update of kPairLambda with X = scale * sum.
// Two launches per iteration replace the 2 + 2 log2(K) of the Smith
// recursion; the sum is the same to rounding.
constexpr int kSeriesX = 0, kSeriesLambda = 1;
constexpr int kSeriesMaxLevels = 5;      // at most K = 2^5 terms as a series
// acceptance: ||A^h||_inf = max row sum |A^h| <= this, h = 2^(J-1); A^h is
// symmetric, so rho^h = ||A^h||_2 <= ||A^h||_inf and the truncated series' tail,
// at most rho^(4h)/(1-rho^2) of X0, is below 1.6e-11 of it
constexpr double kAcceptPower = 2.0e-3;
constexpr double kSelectPower = 4.0e-4;  // level choice: estimated rho^h <= this (5x inside)

struct SeriesArgs {
  int n;
  const double *P;             // K stacked n x n row-major matrices P_k
  const double *G;             // GAMN
  double *part;                // K stacked terms P_k G P_k^T
  const double *bmax;          // block maxima of |GAMN| (k_gemm_pair<kPairGamma>)
  int nbmax;
  double tol;
};

struct SumArgs {
  int n, nterm;
  const double *part;
  double scale;
  double *out;
  const double *occ, *lam;     // kSeriesLambda
  const double *bmax;          // block maxima of |GAMN| (k_gemm_pair<kPairGamma>)
  int nbmax;
  double tol;
  int it;
  const double *pred;          // first iteration: acceptance maxima of the preparation (2 per block)
  int npred;
  double ptol_res, ptol_pow;   // n max|(B+qI)X - I| and n max|A^(2^(J-1))| bounds
  int n_check;                 // n
};

// The convergence test of iteration it (src/paw_waves2.f90:1960-1975) from
// the block maxima of |GAMN|, by the 256 threads of a workgroup: every
// workgroup reaches the same decision; the first one records it.  In the first
// iteration also the acceptance test of the preparation (spectral bounds and
// the Newton-Schulz inverse); a rejection (code 3) makes the host recompute
// the bounds.  True when the loop ends here.
__device__ inline bool series_ends(const SumArgs &a, OrthoState *st) {
  __shared__ double wm[4], wp2[4];
  __shared__ int wn[4];
  double m = 0.0;
  int nan = 0;
  for (int b = threadIdx.x; b < a.nbmax; b += 256) {
    const double x = a.bmax[b];
    if (x != x) nan = 1;
    else m = fmax(m, x);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    m = fmax(m, __shfl_xor(m, o));
    nan |= __shfl_xor(nan, o);
  }
  if ((threadIdx.x & 63) == 0) {
    wm[threadIdx.x >> 6] = m;
    wn[threadIdx.x >> 6] = nan;
  }
  __syncthreads();
  m = fmax(fmax(wm[0], wm[1]), fmax(wm[2], wm[3]));
  nan = wn[0] | wn[1] | wn[2] | wn[3];
  bool reject = false;
  if (a.pred) {
    __syncthreads();
    double p1 = 0.0, p2 = 0.0;
    for (int b = threadIdx.x; b < a.npred; b += 256) {
      p1 = nanmax(p1, a.pred[2 * b]);
      p2 = nanmax(p2, a.pred[2 * b + 1]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      p1 = nanmax(p1, __shfl_xor(p1, o));
      p2 = nanmax(p2, __shfl_xor(p2, o));
    }
    if ((threadIdx.x & 63) == 0) {
      wm[threadIdx.x >> 6] = p1;
      wp2[threadIdx.x >> 6] = p2;
    }
    __syncthreads();
    p1 = nanmax(nanmax(wm[0], wm[1]), nanmax(wm[2], wm[3]));
    p2 = nanmax(nanmax(wp2[0], wp2[1]), nanmax(wp2[2], wp2[3]));
    reject = !((double)a.n_check * p1 <= a.ptol_res && p2 <= a.ptol_pow);
  }
  const int code = reject ? 3 : (nan ? 1 : (m < a.tol ? 0 : (m > 1.0e200 ? 2 : -1)));
  if (code < 0) return false;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->code = code;
    if (code == 0) st->iter = a.it;
    st->done = 1;
  }
  return true;
}

// The test, then the sum of the terms and the epilogue.
template <int MODE>
__global__ void __launch_bounds__(256) k_series_sum(SumArgs a, OrthoState *st) {
  if (stopped(st)) return;
  const int n = a.n;
  const size_t n2 = (size_t)n * n;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const bool in = idx < n * n;
  const int i = in ? idx / n : 0, j = in ? idx - i * n : 0;
  const bool swap = MODE == kSeriesLambda && in && a.occ[i] < a.occ[j];
  // element (i,j), or (j,i) where the update takes the transposed element;
  // the loads of the first group of terms go out with those of the block
  // maxima, the adds run in the order k = 0, 1, ...
  const double *src = a.part + (swap ? (size_t)j * n + i : (size_t)i * n + j);
  constexpr int V = 16;
  double v[V];
#pragma unroll
  for (int u = 0; u < V; ++u) v[u] = (in && u < a.nterm) ? src[(size_t)u * n2] : 0.0;
  if (series_ends(a, st)) return;
  if (!in) return;
  double sum = 0.0;
#pragma unroll
  for (int u = 0; u < V; ++u)
    if (u < a.nterm) sum += v[u];
  for (int k0 = V; k0 < a.nterm; k0 += V) {
#pragma unroll
    for (int u = 0; u < V; ++u) v[u] = k0 + u < a.nterm ? src[(size_t)(k0 + u) * n2] : 0.0;
#pragma unroll
    for (int u = 0; u < V; ++u)
      if (k0 + u < a.nterm) sum += v[u];
  }
  const double c = a.scale * sum;
  if (MODE == kSeriesX) {
    a.out[(size_t)i * n + j] = c;
    return;
  }
  const double oi = a.occ[i] + 1.0e-12, oj = a.occ[j] + 1.0e-12;
  if (swap) {
    const double lt = a.lam[(size_t)j * n + i] - 2.0 * oj / (oj + oi) * c;
    a.out[(size_t)i * n + j] = lt * oi / oj;
  } else {
    a.out[(size_t)i * n + j] = a.lam[(size_t)i * n + j] - 2.0 * oi / (oi + oj) * c;
  }
}

__global__ void k_symm(int n, const double *B, double *Bs) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * n) return;
  const int i = idx / n, j = idx % n;
  Bs[idx] = 0.5 * (B[(size_t)i * n + j] + B[(size_t)j * n + i]);
}

// over the wave: inside the rows of 16 lanes by DPP, across them by two shuffles
__device__ inline double wave_sum(double s) {
  s = row16_sum(s);
  s += __shfl_xor(s, 16);
  return s + __shfl_xor(s, 32);
}

// ---------------------------------------------------------------------------
// Row-panel chains: a workgroup carries a panel of 4, 8 or 16 rows through two or
// more products, the panel between them in LDS.  v_mfma_f64_4x4x4 (4 rows x 16
// columns x 4 k, 16 cycles) splits a matrix into two to four times as many
// workgroups as v_mfma_f64_16x16x4 does at the same rate per cycle; what bounds
// them is the other operand, n^2 doubles per workgroup from the L2 (3.3 us per
// product for 144 bands, of 1.0 for the matrix instructions).  Staging that
// operand through LDS, and splitting the k range over the waves, both came out
// slower.
//   k_series_terms  (P_k G) P_k, 8 or 16 rows, against 16 rows with 16x16x4: 15.8
//                   -> 11.0 us per iteration for 144 bands and 8 terms (16 rows
//                   filled 72 of 256 CUs), 8.0 -> 4.8 for 48, 39.8 -> 24.8 for
//                   256, 88.6 -> 73.0 for 400, 157 -> 117 for 500
//   k_ns_chain      one Newton-Schulz step, X' = 2X - (X (B + qI)) X: 144 bands
//                   9.1 us against 11.4 for its two products as launches
//   k_build_chain   P_k = M A^k, k < K, and the acceptance maxima: 144 bands,
//                   K = 8: 32 us against 41 for the doubling launches
// ---------------------------------------------------------------------------
constexpr int kChainThreads = 1024;
inline int chain_threads(int n) { return 64 * std::min(16, (n + T16 - 1) / T16); }
// LDS row length of a panel: whole groups of eight k and four doubles more, 8 or
// 24 (mod 32) banks, so that the 16-byte reads of (k, k + 1) in the four rows of
// a fragment fall into distinct banks.  With whole rows 8 or 24 (mod 32) doubles
// long every other LDS cycle was a conflict: passes of 16 rows took 87.7 us instead of
// 73.0 for 400 bands and 8 terms, of 8 rows 26.9 instead of 24.8 for 256.
__host__ __device__ inline int chain_ld(int n) {
  return ((n + 7) & ~7) + 4;
}

// acc[f] += A(4f + i, :) B(:, col), the panel A in LDS (columns n .. zero);
// lane l holds A row l % 4 and B column l % 16 at k pair l / 16, and of the
// result row l / 16 and column l % 16.  op(k, value) maps the elements of B.
template <int F, class Op>
__device__ inline void chain_mul(const double *As, int ld, const double *__restrict__ B, int n, int col, double *acc,
                                 Op &&op) {
  constexpr int U = 6;                          // k pairs in flight: 12 loads
  const int lane = threadIdx.x & 63, kq = 2 * (lane >> 4);
  const double *ap = As + (lane & 3) * ld + kq;
  const double *bp = B + min(col, n - 1);
  const int full = n / 8;                       // groups of eight k inside the matrix
  double alt[F];
#pragma unroll
  for (int f = 0; f < F; ++f) alt[f] = 0.0;
  auto step = [&](int p, double b0, double b1) {
    b0 = op(8 * p + kq, b0);
    b1 = op(8 * p + kq + 1, b1);
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const double *q = ap + 4 * f * ld + 8 * p;
      const double a0 = q[0], a1 = q[1];
      acc[f] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, b0, acc[f], 0, 0, 0);
      alt[f] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, b1, alt[f], 0, 0, 0);
    }
  };
  int p = 0;
  for (; p + U <= full; p += U) {
    double b[2 * U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double *r = bp + (size_t)(8 * (p + u) + kq) * n;
      b[2 * u] = r[0];
      b[2 * u + 1] = r[n];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) step(p + u, b[2 * u], b[2 * u + 1]);
  }
  // the remaining groups, rows clamped (their A columns are zero)
  for (; 8 * p < n; p += 2) {
    double b[4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = 8 * (p + u) + kq;
      b[2 * u] = bp[(size_t)min(k, n - 1) * n];
      b[2 * u + 1] = bp[(size_t)min(k + 1, n - 1) * n];
    }
    step(p, b[0], b[1]);
    if (8 * (p + 1) < n) step(p + 1, b[2], b[3]);
  }
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] += alt[f];
}
struct ChainId {
  __device__ double operator()(int, double v) const { return v; }
};
// f(col, column in range) for the column tiles of a wave
template <class F>
__device__ inline void chain_cols(int n, F &&f) {
  const int nt = (n + T16 - 1) / T16, nw = blockDim.x >> 6;
  for (int ct = threadIdx.x >> 6; ct < nt; ct += nw) f(16 * ct + (int)(threadIdx.x & 15));
}
// rows I0 .. I0 + R - 1 of M into LDS, zero outside
template <int R>
__device__ inline void chain_stage(const double *M, int n, int I0, double *s, int ld) {
  for (int e = threadIdx.x; e < R * ld; e += blockDim.x) {
    const int r = e / ld, k = e - r * ld;
    s[e] = (k < n && I0 + r < n) ? M[(size_t)(I0 + r) * n + k] : 0.0;
  }
}

// X' = 2X - U X, U = X (B + qI) of four rows; U is kept for the residual of
// the last step ((B + qI) X is its transpose)
__global__ void __launch_bounds__(kChainThreads) k_ns_chain(int n, double q, const double *Bs, const double *X,
                                                            double *Xn, double *Uo) {
  extern __shared__ double sm[];
  const int ld = chain_ld(n), I0 = blockIdx.x * 4, row = (threadIdx.x & 63) >> 4;
  double *sx = sm, *su = sm + 4 * ld;
  chain_stage<4>(X, n, I0, sx, ld);
  for (int e = threadIdx.x; e < 4 * ld; e += blockDim.x) su[e] = 0.0;
  __syncthreads();
  chain_cols(n, [&](int col) {
    double acc[1] = {0.0};
    chain_mul<1>(sx, ld, Bs, n, col, acc, ChainId{});
    if (col >= n) return;
    const double u = acc[0] + q * sx[row * ld + col];
    su[row * ld + col] = u;
    if (I0 + row < n) Uo[(size_t)(I0 + row) * n + col] = u;
  });
  __syncthreads();
  chain_cols(n, [&](int col) {
    double acc[1] = {0.0};
    chain_mul<1>(su, ld, X, n, col, acc, ChainId{});
    if (col < n && I0 + row < n) Xn[(size_t)(I0 + row) * n + col] = 2.0 * sx[row * ld + col] - acc[0];
  });
}

// P_k = M A^k for 1 <= k < K, A = I - 2qM, four rows of M and of A carried
// through all k (they share the loads of A); the acceptance maxima of these
// rows: max |U - I| and the row sums of |A^h|, h = K/2
__global__ void __launch_bounds__(kChainThreads) k_build_chain(int n, int K, double q, double *P, const double *U,
                                                               double *pred) {
  extern __shared__ double sm[];
  __shared__ double red[2 * kChainThreads / 64];
  const int ld = chain_ld(n), I0 = blockIdx.x * 4, row = (threadIdx.x & 63) >> 4;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const size_t n2 = (size_t)n * n;
  double *cur = sm, *nxt = sm + 8 * ld;
  double r1 = 0.0, r2 = 0.0;
  for (int e = threadIdx.x; e < 4 * ld; e += blockDim.x) {
    const int r = e / ld, k = e - r * ld, i = I0 + r;
    const bool in = k < n && i < n;
    const double m = in ? P[(size_t)i * n + k] : 0.0;
    cur[e] = m;
    cur[4 * ld + e] = in ? (i == k ? 1.0 : 0.0) - 2.0 * q * m : 0.0;
    nxt[e] = 0.0;
    nxt[4 * ld + e] = 0.0;
    if (in) r1 = nanmax(r1, fabs(U[(size_t)i * n + k] - (i == k ? 1.0 : 0.0)));
  }
  __syncthreads();
  for (int k = 1; k <= K; ++k) {
    if (2 * k == K) {                           // cur holds the rows of A^k
      for (int r = wv; r < 4; r += nw) {
        double s = 0.0;
        for (int j = lane; j < n; j += 64) s += fabs(cur[(4 + r) * ld + j]);
        r2 = nanmax(r2, wave_sum(s));
      }
    }
    if (k == K) break;
    double *Pk = P + (size_t)k * n2;
    chain_cols(n, [&](int col) {
      double acc[2] = {0.0, 0.0};
      chain_mul<2>(cur, ld, P, n, col, acc,
                   [&](int kk, double m) { return (kk == col ? 1.0 : 0.0) - 2.0 * q * m; });
      if (col >= n) return;
      nxt[row * ld + col] = acc[0];
      nxt[(4 + row) * ld + col] = acc[1];
      if (I0 + row < n) Pk[(size_t)(I0 + row) * n + col] = acc[0];
    });
    __syncthreads();
    double *s = cur;
    cur = nxt;
    nxt = s;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    r1 = nanmax(r1, __shfl_xor(r1, o));
    r2 = nanmax(r2, __shfl_xor(r2, o));
  }
  if (lane == 0) {
    red[2 * wv] = r1;
    red[2 * wv + 1] = r2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < nw; ++w) {
      r1 = nanmax(r1, red[2 * w]);
      r2 = nanmax(r2, red[2 * w + 1]);
    }
    pred[2 * blockIdx.x] = r1;
    pred[2 * blockIdx.x + 1] = r2;
  }
}

// 4 F rows of the term P_k G P_k (P_k symmetric: the row-major read is the
// coalesced one).  The terms are the fast index of the grid, so that with
// eight of them an XCD reads one P_k.  The convergence test of this iteration
// comes first, as k_series_sum applies it next: when GAMN is converged, NaN or
// diverging the terms go unused and the loop ends there, so the products are
// skipped.  Its loads go out with those of the panel; it costs 0.3 us per
// iteration and saves most of the last one (8 rows): all passes of a solve of 12
// iterations 130 -> 127 us for 144 bands and 8 terms, of 14 iterations 355 -> 339
// for 256; 96 bands 79 -> 77, 48 bands 49 -> 50.  After the first product
// instead of before it, 256 bands took 351.
template <int F>
__global__ void __launch_bounds__(kChainThreads) k_series_terms(SeriesArgs a, int nterm, OrthoState *st) {
  if (stopped(st)) return;
  extern __shared__ double sm[];
  __shared__ int wflag[kChainThreads / 64];
  const int n = a.n, ld = chain_ld(n), row = (threadIdx.x & 63) >> 4;
  const size_t n2 = (size_t)n * n;
  constexpr int R = 4 * F;
  double *sp = sm, *su = sm + R * ld;
  const int k = blockIdx.x % nterm, I0 = R * (blockIdx.x / nterm);
  const double *Pk = a.P + (size_t)k * n2;
  double *out = a.part + (size_t)k * n2;
  const double x0 = (int)threadIdx.x < a.nbmax ? a.bmax[threadIdx.x] : 0.0;
  chain_stage<R>(Pk, n, I0, sp, ld);
  for (int e = threadIdx.x; e < R * ld; e += blockDim.x) su[e] = 0.0;
  bool isnan = false, above = false, huge = false;
  auto test = [&](double x) {
    isnan |= x != x;
    above |= !(x < a.tol);
    huge |= x > 1.0e200;
  };
  test(x0);
  for (int b = threadIdx.x + blockDim.x; b < a.nbmax; b += blockDim.x) test(a.bmax[b]);
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int mine = (__any(isnan) ? 1 : 0) | (__any(above) ? 2 : 0) | (__any(huge) ? 4 : 0);
  if (lane == 0) wflag[threadIdx.x >> 6] = mine;
  __syncthreads();
  const int flag = lane < nw ? wflag[lane] : 0;
  if (__any(flag & 5) || !__any(flag & 2)) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->passes++;
  chain_cols(n, [&](int col) {
    double acc[F] = {};
    chain_mul<F>(sp, ld, a.G, n, col, acc, ChainId{});
    if (col >= n) return;
#pragma unroll
    for (int f = 0; f < F; ++f) su[(4 * f + row) * ld + col] = acc[f];
  });
  __syncthreads();
  chain_cols(n, [&](int col) {
    double acc[F] = {};
    chain_mul<F>(su, ld, Pk, n, col, acc, ChainId{});
    if (col >= n) return;
#pragma unroll
    for (int f = 0; f < F; ++f)
      if (I0 + 4 * f + row < n) out[(size_t)(I0 + 4 * f + row) * n + col] = acc[f];
  });
}

// number of eigenvalues below x of the symmetric tridiagonal (al, be[1..k-1])
__device__ int sturm_count(int k, const double *al, const double *be, double x) {
  int cnt = 0;
  double d = 1.0;
  for (int i = 0; i < k; ++i) {
    d = (al[i] - x) - (i > 0 ? be[i] * be[i] / d : 0.0);
    if (fabs(d) < 1.0e-300) d = -1.0e-300;
    if (d < 0.0) ++cnt;
  }
  return cnt;
}

// Extreme eigenvalues of the symmetric n x n matrix B (row-major) by m-step
// Lanczos with two passes of classical Gram-Schmidt against all previous
// vectors, then multisection on the Sturm sequence of the tridiagonal matrix.
// out = {smallest, largest} Ritz value (inner bounds of the spectrum).
// One workgroup of kLzThreads; the Krylov basis lives in LDS.  What bounds a
// step is B from the L2 into one CU: 16-byte loads of two columns per lane, a
// wave contiguous, sixteen rows in flight (8-byte loads, eight in flight:
// 409 us for 256 bands and 30 steps, now 258; 144 bands 264 -> 192, 500 1057 -> 589).
__global__ void __launch_bounds__(kLzThreads) k_lanczos(int n, int m, const double *__restrict__ B,
                                                        double *out) {
  extern __shared__ double sm[];
  double *V = sm;                          // [m+1][n]
  double *w = V + (size_t)(m + 1) * n;     // [n]
  double *wp = w + n;                      // [G][n] partial matvec, G*n <= 2 kLzThreads
  double *c = wp + 2 * kLzThreads;         // [m+1]
  double *al = c + (m + 1);                // [m]
  double *be = al + m;                     // [m+1]
  __shared__ double red[kLzThreads / 64];
  __shared__ int kend_s;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  constexpr int NW = kLzThreads / 64;
  const int np = (n + 1) / 2, G = min(16, kLzThreads / np);   // column pairs, row groups
  auto block_sum = [&](double s) -> double {
    s = wave_sum(s);
    if (lane == 0) red[wv] = s;
    __syncthreads();
    double r = 0.0;
    for (int q = 0; q < NW; ++q) r += red[q];
    __syncthreads();
    return r;
  };
  double s = 0.0;
  for (int i = t; i < n; i += kLzThreads) {
    const double v = 1.0 + 0.37 * sin(1.7 * i + 0.3);
    V[i] = v;
    s += v * v;
  }
  const double nrm = sqrt(block_sum(s));
  for (int i = t; i < n; i += kLzThreads) V[i] /= nrm;
  if (t == 0) kend_s = m;
  __syncthreads();
  for (int k = 0; k < m; ++k) {
    const double *v = V + (size_t)k * n;
    // w = B v (B symmetric: column reads are coalesced); G row groups per
    // column pair; the last pair of an odd n starts one column earlier
    if (t < G * np) {
      const int p = t % np, g = t / np, col = min(2 * p, n - 2);
      const int jlo = (int)((long)n * g / G), jhi = (int)((long)n * (g + 1) / G);
      double a0 = 0.0, a1 = 0.0, c0 = 0.0, c1 = 0.0;
      int j = jlo;
      auto rows = [&](auto nu) {
        constexpr int U = decltype(nu)::value;
        for (; j + U <= jhi; j += U) {
          dbl2u b[U];
#pragma unroll
          for (int u = 0; u < U; ++u) b[u] = *reinterpret_cast<const dbl2u *>(B + (size_t)(j + u) * n + col);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            double &s0 = u & 1 ? c0 : a0, &s1 = u & 1 ? c1 : a1;
            s0 += b[u].x * v[j + u];
            s1 += b[u].y * v[j + u];
          }
        }
      };
      rows(std::integral_constant<int, 16>{});
      rows(std::integral_constant<int, 4>{});
      rows(std::integral_constant<int, 1>{});
      a0 += c0;
      a1 += c1;
      if (col == 2 * p) wp[g * n + col] = a0;
      wp[g * n + col + 1] = a1;
    }
    __syncthreads();
    for (int i = t; i < n; i += kLzThreads) {
      double r[2] = {0.0, 0.0};
#pragma unroll
      for (int g = 0; g < 16; ++g)
        if (g < G) r[g & 1] += wp[g * n + i];
      w[i] = r[0] + r[1];
    }
    __syncthreads();
    for (int pass = 0; pass < 2; ++pass) {
      for (int j = wv; j <= k; j += NW) {
        double d = 0.0;
        for (int i = lane; i < n; i += 64) d += w[i] * V[(size_t)j * n + i];
        d = wave_sum(d);
        if (lane == 0) c[j] = d;
      }
      __syncthreads();
      if (pass == 0 && t == 0) al[k] = c[k];
      for (int i = t; i < n; i += kLzThreads) {
        double r[4] = {w[i], 0.0, 0.0, 0.0};
        int j = 0;
        for (; j + 3 <= k; j += 4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) r[u] -= c[j + u] * V[(size_t)(j + u) * n + i];
        }
        for (; j <= k; ++j) r[0] -= c[j] * V[(size_t)j * n + i];
        w[i] = (r[0] + r[1]) + (r[2] + r[3]);
      }
      __syncthreads();
    }
    s = 0.0;
    for (int i = t; i < n; i += kLzThreads) s += w[i] * w[i];
    const double b = sqrt(block_sum(s));
    if (t == 0) be[k + 1] = b;
    if (b < 1.0e-14 * fabs(al[k]) || k + 1 == m) {
      if (t == 0) kend_s = k + 1;
      break;
    }
    for (int i = t; i < n; i += kLzThreads) V[(size_t)(k + 1) * n + i] = w[i] / b;
    __syncthreads();
  }
  __syncthreads();
  const int kend = kend_s;
  if (wv > 1) return;
  // wave 0 the smallest, wave 1 the largest eigenvalue: Gershgorin interval of
  // the tridiagonal matrix (every lane)
  double glo = 1.0e300, ghi = -1.0e300;
  for (int i = 0; i < kend; ++i) {
    const double r = (i > 0 ? fabs(be[i]) : 0.0) + (i + 1 < kend ? fabs(be[i + 1]) : 0.0);
    glo = fmin(glo, al[i] - r);
    ghi = fmax(ghi, al[i] + r);
  }
  // multisection: each round splits the bracket into 65 parts, one lane per point
  const int side = wv;
  double lo = glo, hi = ghi;
  for (int round = 0; round < 9; ++round) {
    const double x = lo + (hi - lo) * (double)(lane + 1) / 65.0;
    const int cnt = sturm_count(kend, al, be, x);
    // side 0: smallest eigenvalue = first point with count >= 1
    // side 1: largest eigenvalue = first point with count >= kend
    const bool above = side == 0 ? cnt >= 1 : cnt >= kend;
    const unsigned long long mask = __ballot(above);
    const int first = mask ? __ffsll((long long)mask) - 1 : 64;
    const double nlo = lo + (hi - lo) * (double)first / 65.0;
    const double nhi = lo + (hi - lo) * (double)(first + 1) / 65.0;
    lo = nlo;
    hi = nhi;
  }
  if (lane == 0) out[side] = 0.5 * (lo + hi);
}

// Acceptance test of the spectral bounds (before the outer loop): the
// Newton-Schulz residual R = (B+qI)X - I of the last step (the returned M has
// residual R^2) must be small and so must the last power A^(2^(J-1)), so that
// the truncated series is exact to rounding; otherwise code 3 makes the host
// recompute the bounds.  k_prep_part: one wave per row i forms max_j |R(i,j)|
// and the row sum sum_j |A^h(i,j)|, a workgroup (4 rows) their maxima (NaN
// propagates); the first iteration's k_series_sum decides.
__global__ void __launch_bounds__(256) k_prep_part(int n, const double *T, const double *AJ, double *bmax) {
  __shared__ double r1[4], r2[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int i = blockIdx.x * 4 + wv;
  double m1 = 0.0, s2 = 0.0;
  if (i < n) {
    for (int j = lane; j < n; j += 64) {
      m1 = nanmax(m1, fabs(T[(size_t)i * n + j] - (i == j ? 1.0 : 0.0)));
      s2 += fabs(AJ[(size_t)i * n + j]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    m1 = nanmax(m1, __shfl_xor(m1, o));
    s2 += __shfl_xor(s2, o);
  }
  if (lane == 0) {
    r1[wv] = m1;
    r2[wv] = s2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    bmax[2 * blockIdx.x] = nanmax(nanmax(r1[0], r1[1]), nanmax(r1[2], r1[3]));
    bmax[2 * blockIdx.x + 1] = nanmax(nanmax(r2[0], r2[1]), nanmax(r2[2], r2[3]));
  }
}

__global__ void k_copy_d(size_t n, const double *src, double *dst) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// First Newton-Schulz step from X0 = c I, in closed form:
// X1 = 2 X0 - X0 (B + qI) X0 = 2c I - c^2 (B + qI); also resets the loop state
__global__ void k_ns_first(int n, double c, double q, const double *Bs, double *X, OrthoState *st) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx == 0) {
    st->done = 0;
    st->iter = 0;
    st->code = 0;
    st->passes = 0;
  }
  if (idx >= n * n) return;
  const bool d = idx / n == idx % n;
  X[idx] = (d ? 2.0 * c : 0.0) - c * c * (Bs[idx] + (d ? q : 0.0));
}

// A = I - 2 q M
__global__ void k_cayley(int n, double q, const double *M, double *A) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * n) return;
  A[idx] = ((idx / n == idx % n) ? 1.0 : 0.0) - 2.0 * q * M[idx];
}

// ---------------------------------------------------------------------------
// S^-1 through the eigenvectors of B = sym(CHIPSI), as the reference applies
// it (src/paw_waves2.f90:1889, 1956-1991: LIB$DIAGR8, then
// U[(U^T G U)_ij/(e_i + e_j)]U^T), for a B that is not positive definite,
// where the Cayley series does not converge.
// One workgroup diagonalises B by cyclic Jacobi rotations in the parallel
// round-robin order: each round rotates n/2 disjoint index pairs, A <- J^T A J
// (columns, then rows) and U <- U J; sweeps of n-1 rounds until the
// off-diagonal part is below 1e-15 of the diagonal in the Frobenius norm.
// A (n x n, row-major, overwritten), U[i n + k] = component i of vector k.
constexpr int kJacThreads = 1024;
constexpr int kJacMaxSweeps = 60;
__global__ void __launch_bounds__(kJacThreads) k_jacobi_eig(int n, double *A, double *U, double *e,
                                                            OrthoState *st) {
  __shared__ int sp[kJacThreads], sq[kJacThreads];
  __shared__ double sc[kJacThreads], ss[kJacThreads];
  __shared__ double red[2][kJacThreads / 64];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int m = n + (n & 1);         // players of the round robin; index n is a bye for odd n
  const int np = m / 2;
  for (int idx = t; idx < n * n; idx += kJacThreads) U[idx] = (idx / n == idx % n) ? 1.0 : 0.0;
  if (t == 0) {
    st->done = 0;
    st->iter = 0;
    st->code = 0;
    st->passes = 0;
  }
  __syncthreads();
  for (int sweep = 0; sweep < kJacMaxSweeps; ++sweep) {
    double off = 0.0, dia = 0.0;
    for (int idx = t; idx < n * n; idx += kJacThreads) {
      const double a = A[idx];
      if (idx / n == idx % n) dia += a * a;
      else off += a * a;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      off += __shfl_xor(off, o);
      dia += __shfl_xor(dia, o);
    }
    if (lane == 0) {
      red[0][wv] = off;
      red[1][wv] = dia;
    }
    __syncthreads();
    off = 0.0;
    dia = 0.0;
    for (int w = 0; w < kJacThreads / 64; ++w) {
      off += red[0][w];
      dia += red[1][w];
    }
    __syncthreads();
    if (!(off > 1.0e-30 * dia)) break;   // the same decision in every thread
    for (int r = 0; r < m - 1; ++r) {
      // pairs of round r: (m-1, r) and ((r+k) mod (m-1), (r-k) mod (m-1)), k = 1..np-1
      for (int k = t; k < np; k += kJacThreads) {
        int p = k == 0 ? m - 1 : (r + k) % (m - 1);
        int q = k == 0 ? r : (r - k + (m - 1)) % (m - 1);
        if (p > q) {
          const int x = p;
          p = q;
          q = x;
        }
        double c = 1.0, s = 0.0;
        if (q < n) {
          const double apq = A[(size_t)p * n + q];
          if (apq != 0.0) {
            const double th = (A[(size_t)q * n + q] - A[(size_t)p * n + p]) / (2.0 * apq);
            const double tt = (th >= 0.0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
            c = 1.0 / sqrt(tt * tt + 1.0);
            s = tt * c;
          }
        } else {
          q = p;   // the bye: no rotation
        }
        sp[k] = p;
        sq[k] = q;
        sc[k] = c;
        ss[k] = s;
      }
      __syncthreads();
      // A <- A J and U <- U J: columns p, q of every row
      for (int idx = t; idx < np * n; idx += kJacThreads) {
        const int k = idx / n, i = idx - k * n;
        const int p = sp[k], q = sq[k];
        if (p == q) continue;
        const double c = sc[k], s = ss[k];
        double *ar = A + (size_t)i * n;
        const double ap = ar[p], aq = ar[q];
        ar[p] = c * ap - s * aq;
        ar[q] = s * ap + c * aq;
        double *ur = U + (size_t)i * n;
        const double up = ur[p], uq = ur[q];
        ur[p] = c * up - s * uq;
        ur[q] = s * up + c * uq;
      }
      __syncthreads();
      // A <- J^T A: rows p, q
      for (int idx = t; idx < np * n; idx += kJacThreads) {
        const int k = idx / n, j = idx - k * n;
        const int p = sp[k], q = sq[k];
        if (p == q) continue;
        const double c = sc[k], s = ss[k];
        const double ap = A[(size_t)p * n + j], aq = A[(size_t)q * n + j];
        A[(size_t)p * n + j] = c * ap - s * aq;
        A[(size_t)q * n + j] = s * ap + c * aq;
      }
      __syncthreads();
    }
  }
  for (int i = t; i < n; i += kJacThreads) e[i] = A[(size_t)i * n + i];
}

// X_ij <- X_ij / (e_i + e_j)
__global__ void k_eig_scale(int n, const double *e, double *X, const OrthoState *st) {
  if (stopped(st)) return;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * n) return;
  const int i = idx / n, j = idx - i * n;
  X[idx] /= e[i] + e[j];
}

// ---------------------------------------------------------------------------
// The whole solve in one workgroup, for the small sets whose matrices fit in
// LDS: the preparation (Newton-Schulz, the P_k, the acceptance test) and all
// outer iterations.  As a chain the solve is bound by launch latency: 45
// dependent launches for 2 us of matrix instructions per iteration, most of a
// CP step of Si8 (20 bands, 7 iterations).  One launch: 218 us in kernels (430
// with the gaps) -> 44 us, the step 490 -> 325 us.
//
// Eight waves; a product's 16 x 16 tiles go one per wave, operands from LDS,
// all fragments loaded before the first MFMA.  The term P_k G P_k of row block
// I stays in one wave: G P_k(:,I) comes out of the MFMA in the layout in which
// its transpose P_k(I,:) G is the A operand of the second product (G and P_k
// symmetric), so nothing is exchanged between the two, and both read the same
// fragments of P_k.  kSmallSub waves share the terms of a row block; their
// sums are added in order.  The matrices have a compile-time row
// length of 16 NT + 1 and their rows and columns n .. 4 ceil(n/4) - 1 are
// zero: the products need no bounds (what a tile reads beyond that only
// enters elements that are not written).
// ---------------------------------------------------------------------------
constexpr int kSmallThreads = 512, kSmallTiles = 2, kSmallSub = 4;
constexpr int kSmallMats = 6;                   // LDS matrices beside the P_k
// the pad keeps the rows up to 16 NT of the last matrix inside
inline size_t small_lds(int n, int nterm) {
  const int nt = (n + T16 - 1) / T16, ld = T16 * nt + 1, rows = (n + 3) & ~3;
  return ((size_t)(kSmallMats + nterm) * rows * ld + (T16 * nt - rows) * ld + 64) * sizeof(double);
}

struct SmallArgs {
  int n, nterm, nlev, nns, maxiter;
  double c, q;                                  // Newton-Schulz start, Cayley shift
  double tol, ptol_res, ptol_pow;
  const double *chichi, *psipsi, *chipsi, *occ;
  double *lam;                                  // in: the guess, out: the multipliers
};

// the tile (I, J) of A B (TA: A^T B)
template <int NT, bool TA>
__device__ inline dbl4 small_tile(const double *A, const double *B, int n, int I, int J) {
  constexpr int ld = 16 * NT + 1;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  double a[4 * NT], b[4 * NT];
#pragma unroll
  for (int s = 0; s < 4 * NT; ++s) {
    const int k = 4 * s + lk, i = 16 * I + li;
    a[s] = TA ? A[k * ld + i] : A[i * ld + k];
    b[s] = B[k * ld + 16 * J + li];
  }
  dbl4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 4 * NT; ++s)
    if (4 * s < n) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], acc, 0, 0, 0);
  return acc;
}
// f(r, i, j) over the lane's elements of tile (I, J) inside the matrix
template <class F>
__device__ inline void small_each(int n, int I, int J, F &&f) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 16 * I + lk + 4 * r, j = 16 * J + li;
    if (i < n && j < n) f(r, i, j);
  }
}

template <int NT>
__global__ void __launch_bounds__(kSmallThreads) k_ortho_small(SmallArgs a, OrthoState *st) {
  extern __shared__ double sm[];
  constexpr int EL = (256 * NT * NT + kSmallThreads - 1) / kSmallThreads;   // elements per thread
  constexpr int ld = 16 * NT + 1;
  const int n = a.n, rows = (n + 3) & ~3, n2 = rows * ld;
  double *red = sm;                             // 2 per wave
  double *m0 = sm + 64, *m1 = m0 + n2, *m2 = m1 + n2, *m3 = m2 + n2, *m4 = m3 + n2, *m5 = m4 + n2, *P = m5 + n2;
  const int t = threadIdx.x, wv = t >> 6, lane = t & 63, li = lane & 15, lk = lane >> 4;
  const bool on = wv < NT * NT;
  const int I = wv / NT, J = wv % NT;
  auto finish = [&](int code, int iter, int passes) {
    if (t != 0) return;
    st->code = code;
    st->iter = iter;
    st->passes = passes;
    st->done = code >= 0 ? 1 : 0;
  };
  for (int e = t; e < (kSmallMats + a.nterm) * n2 + (16 * NT - rows) * ld; e += kSmallThreads) m0[e] = 0.0;
  __syncthreads();
  // preparation: B + qI in m0, X in m1/m2, T = (B + qI) X in m3
  for (int e = t; e < n * n; e += kSmallThreads) {
    const int i = e / n, j = e - i * n;
    const double b = 0.5 * (a.chipsi[e] + a.chipsi[j * n + i]) + (i == j ? a.q : 0.0);
    m0[i * ld + j] = b;
    m1[i * ld + j] = (i == j ? 2.0 * a.c : 0.0) - a.c * a.c * b;
  }
  __syncthreads();
  double *x = m1, *y = m2;
  for (int k = 1; k < a.nns; ++k) {
    if (on) {
      const dbl4 v = small_tile<NT, false>(m0, x, n, I, J);
      small_each(n, I, J, [&](int r, int i, int j) { m3[i * ld + j] = v[r]; });
    }
    __syncthreads();
    if (on) {
      const dbl4 v = small_tile<NT, false>(x, m3, n, I, J);
      small_each(n, I, J, [&](int r, int i, int j) { y[i * ld + j] = 2.0 * x[i * ld + j] - v[r]; });
    }
    __syncthreads();
    double *s = x;
    x = y;
    y = s;
  }
  // P_0 = M, A = I - 2qM in m4; level l doubles the P_k and squares A
  double *ap = m4, *an = m5;
  for (int e = t; e < n * n; e += kSmallThreads) {
    const int i = e / n, j = e - i * n;
    const double v = x[i * ld + j];
    P[i * ld + j] = v;
    ap[i * ld + j] = (i == j ? 1.0 : 0.0) - 2.0 * a.q * v;
  }
  __syncthreads();
  for (int l = 0; l < a.nlev; ++l) {
    const int half = 1 << l, nprod = half + (l + 1 < a.nlev ? 1 : 0);
    for (int w = wv; w < nprod * NT * NT; w += kSmallThreads / 64) {
      const int k = w / (NT * NT), tl = w - k * NT * NT, ti = tl / NT, tj = tl % NT;
      double *dst = k < half ? P + (half + k) * n2 : an;
      const dbl4 v = small_tile<NT, false>(ap, k < half ? P + k * n2 : ap, n, ti, tj);
      small_each(n, ti, tj, [&](int r, int i, int j) { dst[i * ld + j] = v[r]; });
    }
    __syncthreads();
    if (l + 1 < a.nlev) {
      double *s = ap;
      ap = an;
      an = s;
    }
  }
  {
    // acceptance, as k_prep_part and the first k_series_sum: the residual of
    // the last Newton-Schulz step and the row sums of |A^(2^(J-1))|
    double r1 = 0.0, r2 = 0.0;
    for (int e = t; e < n * n; e += kSmallThreads) {
      const int i = e / n, j = e - i * n;
      r1 = nanmax(r1, fabs(m3[i * ld + j] - (i == j ? 1.0 : 0.0)));
    }
    for (int i = t; i < n; i += kSmallThreads) {
      double s = 0.0;
      for (int j = 0; j < n; ++j) s += fabs(ap[i * ld + j]);
      r2 = nanmax(r2, s);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      r1 = nanmax(r1, __shfl_xor(r1, o));
      r2 = nanmax(r2, __shfl_xor(r2, o));
    }
    if (lane == 0) {
      red[2 * wv] = r1;
      red[2 * wv + 1] = r2;
    }
    __syncthreads();
    for (int w = 0; w < kSmallThreads / 64; ++w) {
      r1 = nanmax(r1, red[2 * w]);
      r2 = nanmax(r2, red[2 * w + 1]);
    }
    if (!((double)n * r1 <= a.ptol_res && r2 <= a.ptol_pow)) {
      finish(3, 0, 0);
      return;
    }
    __syncthreads();
  }
  // outer iterations: LAMBDA in m0, CHICHI in m5, HAUX in m1, T = LAMBDA^T
  // HAUX in m2, GAMN in m3; the partial sums of the terms in m4, m1, m2, m3
  double cp[4] = {0.0, 0.0, 0.0, 0.0}, pp[4] = {0.0, 0.0, 0.0, 0.0};
  if (on)
    small_each(n, I, J, [&](int r, int i, int j) {
      cp[r] = 2.0 * a.chipsi[i * n + j];
      pp[r] = a.psipsi[min(i, j) * n + max(i, j)] - (i == j ? 1.0 : 0.0);
    });
  double fa[EL], fb[EL];                        // the update's factors (src/paw_waves2.f90:1979-2005)
  bool swap[EL];
#pragma unroll
  for (int u = 0; u < EL; ++u) {
    const int e = t + kSmallThreads * u;
    if (e >= n * n) continue;
    const int i = e / n, j = e - i * n;
    m0[i * ld + j] = a.lam[e];
    m5[i * ld + j] = a.chichi[e];
    const double oi = a.occ[i] + 1.0e-12, oj = a.occ[j] + 1.0e-12;
    swap[u] = a.occ[i] < a.occ[j];
    fa[u] = 2.0 * (swap[u] ? oj / (oj + oi) : oi / (oi + oj));
    fb[u] = oi / oj;
  }
  __syncthreads();
  const int rb = wv / kSmallSub, sub = wv % kSmallSub;
  int code = -1, it = 1;
  for (; it <= a.maxiter; ++it) {
    if (on) {
      const dbl4 v = small_tile<NT, false>(m5, m0, n, I, J);
      small_each(n, I, J, [&](int r, int i, int j) { m1[i * ld + j] = v[r] + cp[r]; });
    }
    __syncthreads();
    if (on) {
      const dbl4 v = small_tile<NT, true>(m0, m1, n, I, J);
      small_each(n, I, J, [&](int r, int i, int j) { m2[i * ld + j] = v[r]; });
    }
    __syncthreads();
    // GAMN and the convergence test (src/paw_waves2.f90:1960-1975): NaN, any
    // element at or above the bound, any far above it
    bool isnan = false, above = false, huge = false;
    if (on)
      small_each(n, I, J, [&](int r, int i, int j) {
        const double g = 0.5 * (m2[i * ld + j] + m2[j * ld + i]) + pp[r];
        m3[i * ld + j] = g;
        isnan |= g != g;
        above |= !(fabs(g) < a.tol);
        huge |= fabs(g) > 1.0e200;
      });
    int flags = (__any(isnan) ? 1 : 0) | (__any(above) ? 2 : 0) | (__any(huge) ? 4 : 0);
    if (lane == 0) reinterpret_cast<int *>(red)[wv] = flags;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSmallThreads / 64; ++w) flags |= reinterpret_cast<const int *>(red)[w];
    if (flags != 2) {
      code = (flags & 1) ? 1 : ((flags & 2) ? 2 : 0);
      break;
    }
    // sum_k P_k G P_k: wave (row block, subset of the terms)
    dbl4 out[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) out[q] = dbl4{0.0, 0.0, 0.0, 0.0};
    if (rb < NT) {
      for (int k = sub; k < a.nterm; k += kSmallSub) {
        const double *Pk = P + k * n2;
        double f[NT][4 * NT];                   // P_k(4 s + lk, 16 q + li)
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
          for (int s = 0; s < 4 * NT; ++s) f[q][s] = Pk[(4 * s + lk) * ld + 16 * q + li];
        dbl4 g[NT];                             // (G P_k)(tile u, rb) = (P_k G)(rb, tile u)^T
#pragma unroll
        for (int u = 0; u < NT; ++u) g[u] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4 * NT; ++s) {
          if (4 * s >= n) break;
          double b = f[0][s];
#pragma unroll
          for (int q = 1; q < NT; ++q) b = rb == q ? f[q][s] : b;
#pragma unroll
          for (int u = 0; u < NT; ++u)
            g[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(m3[(16 * u + li) * ld + 4 * s + lk], b, g[u], 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < 4 * NT; ++s) {
          if (4 * s >= n) break;
#pragma unroll
          for (int q = 0; q < NT; ++q)
            out[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(g[s / 4][s % 4], f[q][s], out[q], 0, 0, 0);
        }
      }
    }
    auto put = [&](double *dst) {
#pragma unroll
      for (int q = 0; q < NT; ++q)
        small_each(n, rb, q, [&](int r, int i, int j) { dst[i * ld + j] = out[q][r]; });
    };
    if (rb < NT && sub < kSmallSub - 1) put(sub == 0 ? m4 : (sub == 1 ? m1 : m2));
    __syncthreads();
    if (rb < NT && sub == kSmallSub - 1) put(m3);
    __syncthreads();
    double nl[EL];
#pragma unroll
    for (int u = 0; u < EL; ++u) {
      const int e = t + kSmallThreads * u;
      if (e >= n * n) continue;
      const int i = e / n, j = e - i * n;
      const int o = swap[u] ? j * ld + i : i * ld + j;
      const double c = 2.0 * a.q * (((m4[o] + m1[o]) + m2[o]) + m3[o]);
      const double v = m0[o] - fa[u] * c;
      nl[u] = swap[u] ? v * fb[u] : v;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < EL; ++u) {
      const int e = t + kSmallThreads * u;
      if (e < n * n) m0[e / n * ld + e % n] = nl[u];
    }
    __syncthreads();
  }
  finish(code, it, it - 1);                     // code -1: not converged in maxiter iterations
  if (code == 0)
    for (int e = t; e < n * n; e += kSmallThreads) a.lam[e] = m0[e / n * ld + e % n];
}

struct OrthoWork {
  double *bs, *m0, *m1, *gam, *x0, *x1, *t1, *t2, *lam2, *occ, *red, *bounds;
  double *apow[kMaxLevels];
  double *pstk, *spart;         // Cayley series: P_k and the terms (K n x n each)
  double *pred;                 // acceptance maxima of the preparation (2 per block)
  OrthoState *st;
};

// block-maxima slots: (n^2+255)/256 for the GAMN maxima, (n+3)/4 row groups
// for the acceptance test (k_prep_part)
inline size_t ortho_slots(size_t n) { return std::max((n * n + 255) / 256, (n + 3) / 4); }
inline size_t ortho_need(size_t n) {
  return (9 + kMaxLevels + 2 * ((size_t)1 << kSeriesMaxLevels)) * n * n + n + 4 * ortho_slots(n) + 64;
}

int ortho_work(pw_waveset *ws, OrthoWork &w) {
  const size_t n2 = (size_t)ws->nb * ws->nb;
  const size_t nblk = ortho_slots(ws->nb);
  const size_t kser = (size_t)1 << kSeriesMaxLevels;
  const size_t need = ortho_need(ws->nb);
  if (need > ws->ortho_cap) {
    if (ws->d_ortho) PW_HIP(hipFree(ws->d_ortho));
    ws->d_ortho = nullptr;
    ws->ortho_cap = 0;
    PW_HIP(hipMalloc(&ws->d_ortho, need * sizeof(double)));
    ws->ortho_cap = need;
  }
  // dynamic LDS limit of the panel kernels: the 160 KiB of a CU less the
  // kernel's static LDS, once per process (the attribute is per kernel, not
  // per waveset; set outside any stream capture)
  static std::once_flag lds_once;
  static hipError_t lds_err = hipSuccess;
  std::call_once(lds_once, [] {
    const void *fns[] = {(const void *)k_panel_batch, (const void *)k_series_terms<2>, (const void *)k_series_terms<4>,
                         (const void *)k_ns_chain, (const void *)k_build_chain, (const void *)k_ortho_small<1>,
                         (const void *)k_ortho_small<2>};
    for (const void *f : fns) {
      hipFuncAttributes fa{};
      hipError_t e = hipFuncGetAttributes(&fa, f);
      if (e == hipSuccess)
        e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(kLdsMax - std::min(kLdsMax, (size_t)fa.sharedSizeBytes)));
      if (e != hipSuccess) lds_err = e;
    }
  });
  PW_HIP(lds_err);
  double *p = ws->d_ortho;
  w.bs = p; p += n2; w.m0 = p; p += n2; w.m1 = p; p += n2; w.gam = p; p += n2;
  w.x0 = p; p += n2; w.x1 = p; p += n2; w.t1 = p; p += n2; w.t2 = p; p += n2;
  w.lam2 = p; p += n2;
  for (int j = 0; j < kMaxLevels; ++j) { w.apow[j] = p; p += n2; }
  w.pstk = p; p += kser * n2;
  w.spart = p; p += kser * n2;
  w.occ = p; p += ws->nb;
  w.bounds = p; p += 8;
  w.st = reinterpret_cast<OrthoState *>(p); p += 8;
  w.pred = p; p += 2 * nblk;
  w.red = p;
  return PW_OK;
}

int gemm(pw_waveset *ws, const double *A, int ta, const double *B, int tb, double *C,
         double alpha = 1.0, const double *D = nullptr, double beta = 0.0,
         const OrthoState *st = nullptr) {
  const int n = ws->nb;
  dim3 grid((n + T16 - 1) / T16, (n + T16 - 1) / T16);
  k_gemm<<<grid, 64 * kGemmWaves, 0, ws->stream>>>(n, A, ta, B, tb, C, alpha, D, beta, st);
  return PW_OK;
}

template <int MODE>
void gemm_pair(pw_waveset *ws, const PairArgs &a, OrthoState *st) {
  const dim3 grid((a.n + T16 - 1) / T16, (a.n + T16 - 1) / T16);
  k_gemm_pair<MODE><<<grid, 64 * kGemmWaves, 0, ws->stream>>>(a, st);
}

int panel_batch(pw_waveset *ws, const BatchArgs &a) {
  if (panel_lds(a.n) > kLdsMax) return pw_fail(PW_ERR_UNSUPPORTED, "WAVES_ORTHO_X: NB too large");
  const dim3 grid((a.n + T16 - 1) / T16, a.nz + (a.Bx ? 1 : 0));
  k_panel_batch<<<grid, 64 * kPanelWaves, panel_lds(a.n), ws->stream>>>(a);
  return PW_OK;
}

// LDS of two panels of `rows` rows
inline size_t chain_lds(int n, int rows) { return (size_t)2 * rows * chain_ld(n) * sizeof(double); }
// rows of a workgroup of the terms: 8 while that gives each CU one workgroup at
// most, 16 beyond, which read the other operand half as often (same sums).  8
// terms: 256 bands (256 workgroups of 8 rows) 24.8 us against 31.4, 272 bands
// (272) 49.4 against 39.2, 400 97.6 against 73.0, 600 301 against 262; 16 terms: 96
// bands 11.3 against 11.6, 128 17.3 against 16.9, 144 30.1 against 30.9, 192 40.8
// against 38.4, 256 88.3 against 64.5, 416 379 against 295.
inline int series_rows(int n, int nterm) { return (n + 7) / 8 * nterm > 256 ? 16 : 8; }
void series_terms(pw_waveset *ws, const SeriesArgs &a, int nterm, OrthoState *st) {
  const int f = series_rows(a.n, nterm) / 4, grid = (a.n + 4 * f - 1) / (4 * f) * nterm;
  auto *const terms = f == 4 ? k_series_terms<4> : k_series_terms<2>;
  terms<<<grid, chain_threads(a.n), chain_lds(a.n, 4 * f), ws->stream>>>(a, nterm, st);
}

template <int MODE>
void series_sum(pw_waveset *ws, const SumArgs &a, OrthoState *st) {
  const int nblk = (int)(((size_t)a.n * a.n + 255) / 256);
  k_series_sum<MODE><<<nblk, 256, 0, ws->stream>>>(a, st);
}

int lanczos_bounds(pw_waveset *ws, const double *d_b, double *d_out, double *lo, double *hi) {
  const int n = ws->nb;
  if (n > kLzThreads) return pw_fail(PW_ERR_UNSUPPORTED, "WAVES_ORTHO_X: NB too large");
  // LDS: (m+1) n + n + 2 kLzThreads + 3m + 2 doubles, at most 152 KiB
  const long budget = 152L * 1024 / 8 - n - 2 * kLzThreads - 3 * kLzMaxSteps - 2;
  int m = std::min({n, kLzMaxSteps, (int)(budget / n) - 1});
  if (m < 2) return pw_fail(PW_ERR_UNSUPPORTED, "WAVES_ORTHO_X: NB too large for the Lanczos bounds");
  const size_t lds = ((size_t)(m + 1) * n + n + 2 * kLzThreads + 3 * (size_t)m + 2) * sizeof(double);
  if (lds > 65536)
    PW_HIP(hipFuncSetAttribute((const void *)k_lanczos, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds));
  k_lanczos<<<1, kLzThreads, lds, ws->stream>>>(n, m, d_b, d_out);
  PW_HIP(hipGetLastError());
  double h[2];
  PW_HIP(hipMemcpyAsync(h, d_out, 2 * sizeof(double), hipMemcpyDeviceToHost, ws->stream));
  PW_HIP(hipStreamSynchronize(ws->stream));
  *lo = h[0];
  *hi = h[1];
  return PW_OK;
}

}  // namespace

namespace {

struct OrthoParams {
  double lo, hi, q;
  int nlev;   // J: S^-1 sums 2^J terms
  int nser;   // the first 2^nser of them as a series (nser <= J), the rest by Smith levels
  int nns;    // Newton-Schulz steps
};

// A Newton-Schulz step as one chain of two products instead of two launches: its
// time grows with n^2 on a quarter of the CUs.  The kernels' times cross just
// above 160 bands: the chain takes 8.2 us for 128, 8.6 for 144, 10.0 for 160,
// 11.7 for 176, 12.2 for 192, 14.3 for 208 and 18.4 for 256, the two launches
// 9.7, 10.0, 10.2, 11.1, 10.9, 12.0 and 12.9 and one more gap.
constexpr int kNsChainMaxN = 160;
// The series matrices one after the other, K - 1 products in one launch,
// instead of doubled in J launches: 32 us against 41 for 144 bands, 71 against
// 82 for 256 and 248 against 280 for 500, all with K = 8; with 16 the doubling
// needs one launch more, the chain 8 products.
constexpr int kBuildChainMaxK = 8;

// M, the series matrices P_k = A^k M, the powers A^(2^j) and the acceptance
// test (everything before the outer loop)
int enqueue_prep(pw_waveset *ws, const OrthoWork &w, const OrthoParams &P) {
  const int n = ws->nb;
  const size_t n2 = (size_t)n * n;
  const int nblk = (int)((n2 + 255) / 256);
  const int ls = P.nser;
  // M = (B + qI)^-1 by Newton-Schulz from X0 = c I, c = 2/(lo+hi+2q): the
  // first step in closed form, the others as GEMM pairs; the last step
  // writes M to P_0 and leaves T = (B+qI) X in t1 for the acceptance test
  const double c = 2.0 / (P.lo + P.hi + 2.0 * P.q);
  k_ns_first<<<nblk, 256, 0, ws->stream>>>(n, c, P.q, w.bs, w.m0, w.st);
  double *mc = w.m0, *mn = w.m1;
  for (int k = 1; k < P.nns; ++k) {
    double *dst = (k + 1 == P.nns) ? w.pstk : mn;
    if (n <= kNsChainMaxN) {
      k_ns_chain<<<(n + 3) / 4, chain_threads(n), chain_lds(n, 4), ws->stream>>>(n, P.q, w.bs, mc, dst, w.t1);
    } else {
      gemm(ws, w.bs, 0, mc, 0, w.t1, 1.0, mc, P.q);     // T = (B+qI) X
      gemm(ws, mc, 0, w.t1, 0, dst, -1.0, mc, 2.0);     // X' = 2X - X T
    }
    mn = mc;
    mc = dst;
  }
  if (ls == P.nlev && (1 << ls) <= kBuildChainMaxK) {
    k_build_chain<<<(n + 3) / 4, chain_threads(n), chain_lds(n, 8), ws->stream>>>(n, 1 << ls, P.q, w.pstk, w.t1,
                                                                                 w.pred);
    PW_HIP(hipGetLastError());
    return PW_OK;
  }
  // A = I - 2qM; level j doubles the series, P_{2^j + k} = A^(2^j) P_k for
  // k < 2^j, and squares the power, A^(2^(j+1)) = A^(2^j) A^(2^j)
  k_cayley<<<nblk, 256, 0, ws->stream>>>(n, P.q, mc, w.apow[0]);
  for (int j = 0; j < ls; ++j) {
    BatchArgs b{};
    b.n = n;
    b.nz = 1 << j;
    b.A = w.apow[j];
    b.B = w.pstk;
    b.sb = n2;
    b.C = w.pstk + ((size_t)1 << j) * n2;
    b.sc = n2;
    if (j + 1 < P.nlev) {
      b.Bx = w.apow[j];
      b.Cx = w.apow[j + 1];
    }
    PW_TRY(panel_batch(ws, b));
  }
  for (int j = ls; j + 1 < P.nlev; ++j) gemm(ws, w.apow[j], 0, w.apow[j], 0, w.apow[j + 1]);
  // acceptance maxima; the test itself runs in the first iteration's k_series_sum
  k_prep_part<<<(n + 3) / 4, 256, 0, ws->stream>>>(n, w.t1, w.apow[P.nlev - 1], w.pred);
  return PW_OK;
}

// outer iterations it0..it1 (1-based, src/paw_waves2.f90:1905-2010)
int enqueue_iters(pw_waveset *ws, const OrthoWork &w, const OrthoParams &P, double *const lbuf[2],
                  const double *d_chichi, const double *d_psipsi, const double *d_chipsi, int it0, int it1) {
  const int n = ws->nb, nt = (n + T16 - 1) / T16;
  const double eps = 1.0e-8;
  const int ls = P.nser;
  for (int it = it0; it <= it1; ++it) {
    const double *lam = lbuf[(it - 1) & 1];
    double *lnew = lbuf[it & 1];
    // HAUX = CHICHI LAMBDA + 2 CHIPSI
    gemm(ws, d_chichi, 0, lam, 0, w.t1, 1.0, d_chipsi, 2.0, w.st);
    {
      // T = LAMBDA^T HAUX, GAMN and its block maxima in one launch
      PairArgs g{};
      g.n = n;
      g.A = lam;
      g.ta = 1;
      g.B = w.t1;
      g.alpha = 1.0;
      g.out = w.gam;
      g.psipsi = d_psipsi;
      g.bmax = w.red;
      gemm_pair<kPairGamma>(ws, g, w.st);
    }
    // X = S^-1(GAMN): the series over the first 2^ls terms, then Smith
    // levels X <- X + A_j X A_j for j >= ls; the convergence test runs first
    // in the series sum.  Without a series (ls = 0) the one term M G M is
    // formed by two products.
    if (ls > 0) {
      SeriesArgs sa{};
      sa.n = n;
      sa.P = w.pstk;
      sa.G = w.gam;
      sa.part = w.spart;
      sa.bmax = w.red;
      sa.nbmax = nt * nt;
      sa.tol = eps;
      series_terms(ws, sa, 1 << ls, w.st);
    } else {
      gemm(ws, w.gam, 0, w.pstk, 0, w.t1, 1.0, nullptr, 0.0, w.st);
      gemm(ws, w.pstk, 0, w.t1, 0, w.spart, 1.0, nullptr, 0.0, w.st);
    }
    SumArgs su{};
    su.n = n;
    su.nterm = 1 << ls;
    su.part = w.spart;
    su.scale = 2.0 * P.q;
    su.occ = w.occ;
    su.lam = lam;
    su.bmax = w.red;
    su.nbmax = nt * nt;
    su.tol = eps;
    su.it = it;
    if (it == 1) {
      // Newton-Schulz residuals square per step: n max|R_k| <= 3.16e-6 for
      // the last T = (B+qI) X_k bounds the returned M's residual by 1e-11
      su.pred = w.pred;
      su.npred = (n + 3) / 4;
      su.ptol_res = 3.16e-6;
      su.ptol_pow = kAcceptPower;
      su.n_check = n;
    }
    if (ls == P.nlev) {
      su.out = lnew;
      series_sum<kSeriesLambda>(ws, su, w.st);
      continue;
    }
    su.out = w.x0;
    series_sum<kSeriesX>(ws, su, w.st);
    double *xc = w.x0, *xn = w.x1;
    for (int j = ls; j < P.nlev; ++j) {
      gemm(ws, xc, 0, w.apow[j], 0, w.t1, 1.0, nullptr, 0.0, w.st);
      if (j + 1 < P.nlev) {
        gemm(ws, w.apow[j], 0, w.t1, 0, xn, 1.0, xc, 1.0, w.st);
        std::swap(xc, xn);
      } else {
        // last level: X = A_j T + X and the LAMBDA update in one launch
        PairArgs l{};
        l.n = n;
        l.A = w.apow[j];
        l.B = w.t1;
        l.D = xc;
        l.alpha = 1.0;
        l.beta = 1.0;
        l.out = lnew;
        l.occ = w.occ;
        l.lam = lam;
        gemm_pair<kPairLambda>(ws, l, w.st);
      }
    }
  }
  return PW_OK;
}

// outer iterations it0..it1 with S^-1 from the eigenvectors U (w.m1) and the
// eigenvalues e (w.x1) of B: the reference's own form of the update
int enqueue_iters_eig(pw_waveset *ws, const OrthoWork &w, double *const lbuf[2], const double *d_chichi,
                      const double *d_psipsi, const double *d_chipsi, int it0, int it1) {
  const int n = ws->nb, nt = (n + T16 - 1) / T16;
  const int nblk = (n * n + 255) / 256;
  for (int it = it0; it <= it1; ++it) {
    const double *lam = lbuf[(it - 1) & 1];
    double *lnew = lbuf[it & 1];
    gemm(ws, d_chichi, 0, lam, 0, w.t1, 1.0, d_chipsi, 2.0, w.st);
    {
      PairArgs g{};
      g.n = n;
      g.A = lam;
      g.ta = 1;
      g.B = w.t1;
      g.alpha = 1.0;
      g.out = w.gam;
      g.psipsi = d_psipsi;
      g.bmax = w.red;
      gemm_pair<kPairGamma>(ws, g, w.st);
    }
    gemm(ws, w.m1, 1, w.gam, 0, w.t2, 1.0, nullptr, 0.0, w.st);    // U^T G
    gemm(ws, w.t2, 0, w.m1, 0, w.x0, 1.0, nullptr, 0.0, w.st);     // (U^T G) U
    k_eig_scale<<<nblk, 256, 0, ws->stream>>>(n, w.x1, w.x0, w.st);
    gemm(ws, w.m1, 0, w.x0, 0, w.t2, 1.0, nullptr, 0.0, w.st);     // U (...)
    gemm(ws, w.t2, 0, w.m1, 1, w.spart, 1.0, nullptr, 0.0, w.st);  // (...) U^T
    SumArgs su{};
    su.n = n;
    su.nterm = 1;
    su.part = w.spart;
    su.scale = 1.0;
    su.occ = w.occ;
    su.lam = lam;
    su.bmax = w.red;
    su.nbmax = nt * nt;
    su.tol = 1.0e-8;
    su.it = it;
    su.out = lnew;
    series_sum<kSeriesLambda>(ws, su, w.st);
  }
  PW_HIP(hipGetLastError());
  return PW_OK;
}

// the reference's stop conditions (src/paw_waves2.f90:1935-1945, 1960-1975)
int ortho_status(const OrthoState &hs) {
  if (hs.code == 1) return pw_fail(PW_ERR_NOCONV, "WAVES_ORTHO_X: NaN in overlap");
  if (hs.code == 2)
    return pw_fail(PW_ERR_NOCONV, "WAVES_ORTHO_X: iteration loop for orthogonalization is about to diverge");
  if (!hs.done)
    return pw_fail(PW_ERR_NOCONV,
                   "WAVES_ORTHO_X: loop for orthogonalization is not converged (specify SAFEORTHO=F, "
                   "reduce the cutoff or the time step)");
  return PW_OK;
}

// WAVES_ORTHO_X with S^-1 from the eigenvectors of B (the reference's form),
// for a B that is not positive definite (inside the Lanczos bounds or
// rejected by the series' acceptance test)
int ortho_x_eig(pw_waveset *ws, const OrthoWork &w, double *const lbuf[2], double *d_lam, const double *d_chichi,
                const double *d_psipsi, const double *d_chipsi, int *iter) {
  const int n = ws->nb;
  const size_t n2 = (size_t)n * n;
  const int nblk = (int)((n2 + 255) / 256);
  if (n > 2 * kJacThreads) return pw_fail(PW_ERR_UNSUPPORTED, "WAVES_ORTHO_X: NB too large");
  ws->ortho_eigen++;
  k_copy_d<<<nblk, 256, 0, ws->stream>>>(n2, w.bs, w.m0);
  k_jacobi_eig<<<1, kJacThreads, 0, ws->stream>>>(n, w.m0, w.m1, w.x1, w.st);
  PW_HIP(hipGetLastError());
  int launched = 0;
  OrthoState hs{};
  OrthoState *hp = static_cast<OrthoState *>(ws->h_ortho_state);
  while (launched < kMaxIter) {
    const int nit = std::min(launched == 0 ? 8 : 4, kMaxIter - launched);
    PW_TRY(enqueue_iters_eig(ws, w, lbuf, d_chichi, d_psipsi, d_chipsi, launched + 1, launched + nit));
    launched += nit;
    PW_HIP(hipMemcpyAsync(hp, w.st, sizeof(OrthoState), hipMemcpyDeviceToHost, ws->stream));
    PW_HIP(hipStreamSynchronize(ws->stream));
    hs = *hp;
    if (hs.done) break;
  }
  PW_TRY(ortho_status(hs));
  if ((hs.iter - 1) & 1) {
    k_copy_d<<<nblk, 256, 0, ws->stream>>>(n2, w.lam2, d_lam);
    PW_HIP(hipGetLastError());
  }
  ws->ortho_levels = 0;
  ws->ortho_series = 0;
  ws->ortho_ns = 0;
  *iter = hs.iter;
  return PW_OK;
}

}  // namespace

void ortho_graph_release(pw_waveset *ws) {
  if (ws->ortho_exec) (void)hipGraphExecDestroy((hipGraphExec_t)ws->ortho_exec);
  ws->ortho_exec = nullptr;
}

int ortho_x_device(pw_waveset *ws, double *d_lam, const double *d_chichi, const double *d_psipsi,
                   const double *d_chipsi, int *iter) {
  ScopeTimer tm(ws, "ortho_x");
  const int n = ws->nb;
  const size_t n2 = (size_t)n * n;
  const int nblk = (int)((n2 + 255) / 256);
  OrthoWork w;
  const double *old_base = ws->d_ortho;
  PW_TRY(ortho_work(ws, w));
  if (ws->d_ortho != old_base) ortho_graph_release(ws);
  if (ws->d_occ) w.occ = ws->d_occ;   // the waveset's occupations are on the device already
  else PW_HIP(hipMemcpyAsync(w.occ, ws->occ.data(), n * sizeof(double), hipMemcpyHostToDevice, ws->stream));
  if (!ws->h_ortho_state) PW_HIP(hipHostMalloc(&ws->h_ortho_state, sizeof(OrthoState), hipHostMallocDefault));
  bool have_bs = false;
  auto symm = [&]() -> int {
    if (!have_bs) k_symm<<<nblk, 256, 0, ws->stream>>>(n, d_chipsi, w.bs);
    have_bs = true;
    PW_HIP(hipGetLastError());
    return PW_OK;
  };
  ws->ortho_lanczos = 0;
  ws->ortho_passes = 0;
  double *lbuf[2] = {d_lam, w.lam2};
  for (int attempt = 0; attempt < 2; ++attempt) {
    // spectral bounds of B: inner Ritz bounds, reused from the previous call
    // until the acceptance test rejects them
    if (!ws->lz_valid || attempt > 0) {
      double lo0, hi0;
      PW_TRY(symm());
      PW_TRY(lanczos_bounds(ws, w.bs, w.bounds, &lo0, &hi0));
      ws->lz_lo = lo0;
      ws->lz_hi = hi0;
      ws->lz_valid = true;
      ws->ortho_lanczos++;
    }
    OrthoParams P;
    P.lo = ws->lz_lo;
    P.hi = ws->lz_hi;
    if (!(P.lo > 0.0) || !(P.hi >= P.lo)) {
      // sym(CHIPSI) is not positive definite: the eigenvector form of S^-1
      ws->lz_valid = false;
      PW_TRY(symm());
      return ortho_x_eig(ws, w, lbuf, d_lam, d_chichi, d_psipsi, d_chipsi, iter);
    }
    P.lo *= 0.97;
    P.hi *= 1.03;
    P.q = std::sqrt(P.lo * P.hi);
    const double kap = P.hi / P.lo;
    const double rho = (std::sqrt(kap) - 1.0) / (std::sqrt(kap) + 1.0);
    // S^-1 sums A^k X0 A^k for k < K = 2^J.  The acceptance test certifies
    // h = 2^(J-1) by ||A^h||_inf <= kAcceptPower = 2e-3; then rho^h =
    // ||A^h||_2 <= ||A^h||_inf and the tail, at most rho^(2K)/(1-rho^2) of X0,
    // is below 1.6e-11 of it.  J is the least level count whose estimate from
    // the (widened) Lanczos bounds, rho^h, is 5x inside the test; a second
    // attempt (bounds rejected once) adds a level.
    P.nlev = 1;
    if (rho > 1.0e-300) {
      const double need = std::log(kSelectPower) / std::log(rho);
      P.nlev = std::max(1, (int)std::ceil(std::log2(std::max(need, 1.0))) + 1);
    }
    P.nlev += attempt;
    P.nser = series_fits(n) ? std::min(P.nlev, kSeriesMaxLevels) : 0;
    if (P.nlev > kMaxLevels) {
      ws->lz_valid = false;
      PW_TRY(symm());
      return ortho_x_eig(ws, w, lbuf, d_lam, d_chichi, d_psipsi, d_chipsi, iter);
    }
    // Newton-Schulz for (B+qI)^-1: |I - (B+qI)X_k| = e0^(2^k); stop at 1e-17
    // (the acceptance test asks for 1e-11)
    const double kp = (P.hi + P.q) / (P.lo + P.q);
    const double e0 = (kp - 1.0) / (kp + 1.0);
    P.nns = 2;
    if (e0 > 1.0e-300) P.nns = std::max(2, (int)std::ceil(std::log2(std::max(1.0, std::log(1.0e-17) / std::log(e0)))));
    ws->ortho_levels = P.nlev;
    ws->ortho_series = 1 << P.nser;
    ws->ortho_ns = P.nns;
    OrthoState hs{};
    OrthoState *hp = static_cast<OrthoState *>(ws->h_ortho_state);
    // one workgroup for the whole solve where its matrices fit in LDS and a
    // product has at most four tiles: 32 bands with 8 terms of the series, 24
    // with 16, 16 with 32.  The launches of the chain take 218 us in kernels and 430 with
    // the gaps for 20 bands, this one 44; for 32 bands 230 and 500 against 64.
    // Wider sets do not fit with their 8 terms.
    if (P.nser == P.nlev && (n + T16 - 1) / T16 <= kSmallTiles && small_lds(n, 1 << P.nser) <= kLdsMax) {
      const int nts = (n + T16 - 1) / T16;
      auto *const small = nts == 1 ? k_ortho_small<1> : k_ortho_small<2>;
      SmallArgs s{};
      s.n = n;
      s.nterm = 1 << P.nser;
      s.nlev = P.nlev;
      s.nns = P.nns;
      s.maxiter = kMaxIter;
      s.c = 2.0 / (P.lo + P.hi + 2.0 * P.q);
      s.q = P.q;
      s.tol = 1.0e-8;
      s.ptol_res = 3.16e-6;
      s.ptol_pow = kAcceptPower;
      s.chichi = d_chichi;
      s.psipsi = d_psipsi;
      s.chipsi = d_chipsi;
      s.occ = w.occ;
      s.lam = d_lam;
      (*small)<<<1, kSmallThreads, small_lds(n, s.nterm), ws->stream>>>(s, w.st);
      PW_HIP(hipGetLastError());
      PW_HIP(hipMemcpyAsync(hp, w.st, sizeof(OrthoState), hipMemcpyDeviceToHost, ws->stream));
      PW_HIP(hipStreamSynchronize(ws->stream));
      hs = *hp;
      if (hs.code == 3 && attempt == 0) continue;
      if (hs.code == 3) {
        ws->lz_valid = false;
        PW_TRY(symm());
        return ortho_x_eig(ws, w, lbuf, d_lam, d_chichi, d_psipsi, d_chipsi, iter);
      }
      ws->ortho_passes = hs.passes;
      PW_TRY(ortho_status(hs));
      *iter = hs.iter;
      return PW_OK;
    }
    PW_TRY(symm());
    const int batch = std::max(2, std::min(ws->ortho_iter > 0 ? ws->ortho_iter : 8, kMaxIter));
    // the preparation and the first batch of iterations are one captured graph,
    // replayed while the bounds, the batch and the buffers stay the same
    const OrthoGraphKey key{P.lo, P.hi, P.nlev, P.nns, batch, d_lam, d_chichi, d_psipsi, d_chipsi, ws->d_ortho};
    if (!ws->ortho_exec || !(ws->ortho_key == key)) {
      ortho_graph_release(ws);
      // with other plans or wavesets alive (a request loop), and for a single
      // solve (capture, instantiation and release cost more than the launches
      // of the one replay save), the work is issued directly below; an existing graph is still replayed
      CaptureGate &gate = capture_gate();
      std::unique_lock<std::mutex> lk(gate.mu);
      if (!ws->ortho_once && gate.plans <= 1 && gate.wavesets <= 1) {
        PW_HIP(hipStreamBeginCapture(ws->stream, hipStreamCaptureModeRelaxed));
        int rq = enqueue_prep(ws, w, P);
        if (rq == PW_OK) rq = enqueue_iters(ws, w, P, lbuf, d_chichi, d_psipsi, d_chipsi, 1, batch);
        hipGraph_t graph = nullptr;
        const hipError_t ec = hipStreamEndCapture(ws->stream, &graph);
        const hipError_t el = hipGetLastError();
        if (rq != PW_OK || ec != hipSuccess || el != hipSuccess || !graph) {
          if (graph) (void)hipGraphDestroy(graph);
          if (rq != PW_OK) return rq;
          return pw_fail(PW_ERR_HIP, std::string("WAVES_ORTHO_X: graph capture failed: ") +
                                         hipGetErrorString(ec != hipSuccess ? ec : el));
        }
        hipGraphExec_t exec = nullptr;
        const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ei != hipSuccess)
          return pw_fail(PW_ERR_HIP, std::string("WAVES_ORTHO_X: graph instantiation failed: ") +
                                         hipGetErrorString(ei));
        ws->ortho_exec = exec;
        ws->ortho_key = key;
      }
    }
    if (ws->ortho_exec) {
      PW_HIP(hipGraphLaunch((hipGraphExec_t)ws->ortho_exec, ws->stream));
    } else {
      PW_TRY(enqueue_prep(ws, w, P));
      PW_TRY(enqueue_iters(ws, w, P, lbuf, d_chichi, d_psipsi, d_chipsi, 1, batch));
      PW_HIP(hipGetLastError());
      ws->ortho_graph_misses++;
    }
    int launched = batch;
    for (;;) {
      PW_HIP(hipMemcpyAsync(hp, w.st, sizeof(OrthoState), hipMemcpyDeviceToHost, ws->stream));
      PW_HIP(hipStreamSynchronize(ws->stream));
      hs = *hp;
      if (hs.done || launched >= kMaxIter) break;
      const int nit = std::min(4, kMaxIter - launched);
      PW_TRY(enqueue_iters(ws, w, P, lbuf, d_chichi, d_psipsi, d_chipsi, launched + 1, launched + nit));
      PW_HIP(hipGetLastError());
      launched += nit;
    }
    if (hs.code == 3) {
      if (attempt == 0) continue;
      // bounds rejected twice: B is indefinite or too ill-conditioned for
      // the series; the eigenvector form takes any symmetric B
      ws->lz_valid = false;
      return ortho_x_eig(ws, w, lbuf, d_lam, d_chichi, d_psipsi, d_chipsi, iter);
    }
    ws->ortho_passes = hs.passes;
    PW_TRY(ortho_status(hs));
    // iteration hs.iter converged after hs.iter-1 updates
    if ((hs.iter - 1) & 1) {
      k_copy_d<<<nblk, 256, 0, ws->stream>>>(n2, w.lam2, d_lam);
      PW_HIP(hipGetLastError());
    }
    *iter = hs.iter;
    return PW_OK;
  }
  return pw_fail(PW_ERR_NOCONV, "WAVES_ORTHO_X: spectral bounds of sym(CHIPSI) not accepted");
}

// ---------------------------------------------------------------------------
// C ABI: WAVES_ORTHO_X on host matrices, column-major (pw_ortho_x) or row-major
// (pw_ortho_x_rows) NB x NB.
//
// What bounded the call was the host: transposes by element loops on both
// sides of the C entry (0.9 of 2.1 ms for 256 bands), the creation of a stream,
// a graph that is replayed once.  The matrices are uploaded as they are and
// transposed on the device, the solve runs on the thread's default stream with
// its launches issued directly, all device memory is one allocation.
// ---------------------------------------------------------------------------
namespace {

// out_m = transpose of in_m, m = blockIdx.z, by 32 x 32 tiles
__global__ void __launch_bounds__(256) k_transpose_mats(int n, const double *__restrict__ in,
                                                        double *__restrict__ out) {
  __shared__ double s[32][33];
  const size_t o = (size_t)blockIdx.z * n * n;
  const int i0 = blockIdx.y * 32, j0 = blockIdx.x * 32, c = threadIdx.x & 31, r = threadIdx.x >> 5;
  for (int q = r; q < 32; q += 8)
    if (i0 + q < n && j0 + c < n) s[q][c] = in[o + (size_t)(i0 + q) * n + j0 + c];
  __syncthreads();
  for (int q = r; q < 32; q += 8)
    if (j0 + q < n && i0 + c < n) out[o + (size_t)(j0 + q) * n + i0 + c] = s[c][q];
}

int ortho_x_host(int nb, const double *occ, const double *const src[4], double *lambda, int *iter, bool rows) {
  pw_waveset ws;
  OrthoState state{};
  ws.nb = nb;
  ws.stream = hipStreamPerThread;
  ws.occ.assign(occ, occ + nb);
  ws.h_ortho_state = &state;
  ws.ortho_once = true;
  const size_t n2 = (size_t)nb * nb, need = ortho_need(nb), mats = (rows ? 4 : 8) * n2;
  double *base = nullptr;
  PW_HIP(hipMalloc(&base, (need + mats) * sizeof(double)));
  ws.d_ortho = base;
  ws.ortho_cap = need;
  double *d = base + need, *up = rows ? d : d + 4 * n2;
  const dim3 grid((nb + 31) / 32, (nb + 31) / 32, 4);
  int rc = PW_OK;
  for (int m = 0; m < 4 && rc == PW_OK; ++m)
    if (hipMemcpyAsync(up + m * n2, src[m], n2 * sizeof(double), hipMemcpyHostToDevice, ws.stream) != hipSuccess)
      rc = pw_fail(PW_ERR_HIP, "pw_ortho_x: upload failed");
  if (rc == PW_OK && !rows) {
    k_transpose_mats<<<grid, 256, 0, ws.stream>>>(nb, up, d);
    if (hipGetLastError() != hipSuccess) rc = pw_fail(PW_ERR_HIP, "pw_ortho_x: transposition failed");
  }
  if (rc == PW_OK) rc = ortho_x_device(&ws, d + 3 * n2, d, d + n2, d + 2 * n2, iter);
  if (rc == PW_OK && !rows) {
    k_transpose_mats<<<dim3(grid.x, grid.y, 1), 256, 0, ws.stream>>>(nb, d + 3 * n2, up);
    if (hipGetLastError() != hipSuccess) rc = pw_fail(PW_ERR_HIP, "pw_ortho_x: transposition failed");
  }
  if (rc == PW_OK &&
      hipMemcpyAsync(lambda, rows ? d + 3 * n2 : up, n2 * sizeof(double), hipMemcpyDeviceToHost, ws.stream) != hipSuccess)
    rc = pw_fail(PW_ERR_HIP, "pw_ortho_x: download failed");
  if (hipStreamSynchronize(ws.stream) != hipSuccess && rc == PW_OK)
    rc = pw_fail(PW_ERR_HIP, "pw_ortho_x: stream synchronisation failed");
  (void)hipFree(base);
  return rc;
}

}  // namespace

extern "C" int pw_ortho_x(int nb, const double *occ, const double *chichi, const double *psipsi,
                          const double *chipsi, double *lambda, int *iter) {
  if (nb <= 0 || !occ || !chichi || !psipsi || !chipsi || !lambda || !iter)
    return pw_fail(PW_ERR_ARG, "pw_ortho_x: bad argument");
  const double *const src[4] = {chichi, psipsi, chipsi, lambda};
  return ortho_x_host(nb, occ, src, lambda, iter, false);
}

extern "C" int pw_ortho_x_rows(int nb, const double *occ, const double *chichi, const double *psipsi,
                               const double *chipsi, double *lambda, int *iter) {
  if (nb <= 0 || !occ || !chichi || !psipsi || !chipsi || !lambda || !iter)
    return pw_fail(PW_ERR_ARG, "pw_ortho_x: bad argument");
  const double *const src[4] = {chichi, psipsi, chipsi, lambda};
  return ortho_x_host(nb, occ, src, lambda, iter, true);
}
