// Device helpers shared by the WAVES kernels (pw_kernels.hip, pw_gamma.hip).
#pragma once
#include "pw_common.h"

namespace {

__device__ inline double2 czero() { return make_double2(0.0, 0.0); }

struct ProjGeo {
  int ngl, nbh, nat, lmnxx, nphase, nmaxx;
  const int *igvec;        // 3*ngl
  const double *pro;       // [nbarepro][ngl]
  const double *ylm;       // [lmx][ngl]
  const double2 *phase;    // [nat][3][nphase]
  const int *atom_isp, *ipro0, *ibpro, *lmnx;
  const int *lmn_ln, *lmn_lm, *lmn_l;   // [nsp][lmnxx]
};

__device__ inline double2 eigr_of(const ProjGeo &q, int atom, int ig) {
  const int *iv = q.igvec + 3 * ig;
  const double2 *ph = q.phase + (size_t)atom * 3 * q.nphase;
  double2 e = cmul(ph[iv[0] + q.nmaxx], ph[q.nphase + iv[1] + q.nmaxx]);
  return cmul(e, ph[2 * q.nphase + iv[2] + q.nmaxx]);
}

inline ProjGeo make_pgeo(pw_waveset *ws) {
  ProjGeo q;
  pw_plan *p = ws->plan;
  q.ngl = p->ngl; q.nbh = ws->nbh; q.nat = ws->nat; q.lmnxx = ws->lmnxx;
  q.nphase = ws->nphase; q.nmaxx = (ws->nphase - 1) / 2;
  q.igvec = p->d_igvec; q.pro = ws->d_pro; q.ylm = ws->d_ylm; q.phase = ws->d_phase;
  q.atom_isp = ws->d_atom_isp; q.ipro0 = ws->d_ipro0; q.ibpro = ws->d_ibpro; q.lmnx = ws->d_lmnx;
  q.lmn_ln = ws->d_lmn_ln; q.lmn_lm = ws->d_lmn_lm; q.lmn_l = ws->d_lmn_l;
  return q;
}

// XCD-aware tile order.  Workgroups are dealt to the eight XCDs in turn
// (linear id mod 8), and each XCD has its own L2.  The tiles that read the
// same operand block (one G range) get linear ids of one residue mod 8 that
// follow each other in that XCD's order, so the block is fetched from HBM once
// instead of once per tile.  Grid: xcd_blocks(ninner, nshared) in x.
constexpr int kXcd = 8;
struct XcdTile {
  int inner, shared;
  bool valid;
};
__device__ inline XcdTile xcd_tile(int ninner, int nshared) {
  const int L = blockIdx.x, x = L % kXcd, slot = L / kXcd;
  XcdTile t;
  t.inner = slot % ninner;
  t.shared = (slot / ninner) * kXcd + x;
  t.valid = t.shared < nshared;
  return t;
}
inline unsigned xcd_blocks(int ninner, int nshared) {
  return (unsigned)((nshared + kXcd - 1) / kXcd) * kXcd * ninner;
}

// sum of v over the 16 lanes of a DPP row (lanes 16k .. 16k+15), in every lane
// of the row: four rotate-and-add steps on the cross-lane (DPP) path of the
// VALU (row_ror 8, 4, 2, 1), no LDS traffic
template <int CTRL>
__device__ inline double dpp_ror(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ inline double row16_sum(double v) {
  v += dpp_ror<0x128>(v);
  v += dpp_ror<0x124>(v);
  v += dpp_ror<0x122>(v);
  v += dpp_ror<0x121>(v);
  return v;
}

// z * (-i)^l
__device__ inline double2 rot_mil(double2 z, int l) {
  switch (l & 3) {
    case 0: return z;
    case 1: return make_double2(z.y, -z.x);
    case 2: return make_double2(-z.x, -z.y);
    default: return make_double2(-z.y, z.x);
  }
}

typedef double dbl4 __attribute__((ext_vector_type(4)));

// v_mfma_f64_16x16x4f64: A(i,k) in lane i+16k, B(k,j) in lane j+16k, C(i,j)
// in lane j+16(i%4), element i/4
__device__ inline dbl4 mfma4(double a, double b, dbl4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// sum of split partials: out[i] = scale * sum_s part[s][i] in a fixed order.
// A block takes 32 outputs; its 8 lanes per output stride over the splits
// and are combined through LDS.
constexpr int kRedC = 32, kRedS = 8;

__device__ inline double rz(double) { return 0.0; }
__device__ inline double2 rz(double2) { return make_double2(0.0, 0.0); }
__device__ inline double radd(double a, double b) { return a + b; }
__device__ inline double2 radd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double rscale(double a, double s) { return a * s; }
__device__ inline double2 rscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }

// out[i] = scale * sum_k part[k][i]: kRedS lanes per column take the splits
// k = sl, sl + kRedS, ...; each lane issues its loads 16 at a time and adds
// them in k order, then the lanes are added in order (deterministic)
template <typename T>
__global__ void __launch_bounds__(kRedC * kRedS) k_reduce_split(const T *__restrict__ part, int ns, int n,
                                                                double scale, T *__restrict__ out) {
  __shared__ T red[kRedS][kRedC];
  const int c = threadIdx.x % kRedC, sl = threadIdx.x / kRedC;
  const int i = blockIdx.x * kRedC + c;
  T acc = rz(T());
  if (i < n) {
    constexpr int V = 16;
    for (int k0 = sl; k0 < ns; k0 += V * kRedS) {
      T v[V];
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int k = k0 + u * kRedS;
        v[u] = k < ns ? part[(size_t)k * n + i] : rz(T());
      }
#pragma unroll
      for (int u = 0; u < V; ++u) acc = radd(acc, v[u]);
    }
  }
  red[sl][c] = acc;
  __syncthreads();
  if (sl != 0 || i >= n) return;
  T r = red[0][c];
#pragma unroll
  for (int q = 1; q < kRedS; ++q) r = radd(r, red[q][c]);
  out[i] = rscale(r, scale);
}

}  // namespace
