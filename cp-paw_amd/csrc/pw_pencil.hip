// Pencil passes (y and z) of the full-grid transforms for lengths fixed at
// compile time.
//
// HBM bound: the z pass of 128 transforms of 64^3 in FP64 reads 226 MB and
// writes 537 MB in 130 us (5.9 TB/s; the planes that the y pass has just written
// come in part from the last-level cache), 113 us for a kernel that only loads
// and stores in this pattern.  The first stage takes its radix-R inputs straight from global
// memory into registers and the last stage writes its outputs straight back,
// so LDS holds only the exchange between stages and a thread has R
// independent loads in flight; pencils of the z pass are the flat (y, x)
// index, so a tile's rows are TP contiguous elements whatever NR1 is.
// Measured there against whole transforms in two LDS buffers with run-time
// lengths: z 274 -> 130 us, y 88 -> 45, the x pass with its stripes as rows
// 41 -> 25; with 72^3 x 90, z 320 -> 145 and y 135 -> 55 us.  Loads in
// branches of their own (absent rows) had made the z pass 248 us.
#include "pw_dft.h"
#include "pw_pencil.h"

namespace {

constexpr int kPB = 256;

// Stages of a pencil transform: the run-time kernel's in FP32 (the same
// rounding for every length, with or without an instantiation here); in FP64
// a factor 64 or 32 goes as 8 8 or 8 4 instead of 16 4 or 16 2, which keeps
// all threads of the first stage busy with half the registers.
template <typename T2>
__host__ __device__ constexpr Fft1D pencil_stages(int n) {
  Fft1D f = fft_stockham_ct(n);
  if (sizeof(T2) == sizeof(double2) && f.nstage >= 2 && f.radix[f.nstage - 2] == 16 && f.radix[f.nstage - 1] <= 4) {
    f.radix[f.nstage - 2] = 8;
    f.radix[f.nstage - 1] *= 2;
  }
  return f;
}

// pencils per workgroup.  Narrow tiles, 16 pencils (128-byte rows in FP32, 256 in
// FP64), fill the chip where a pass has few pencils and waste few lanes where
// NR1 is no multiple of a wide tile (the y pass has NR1 pencils per plane).  Wide
// ones, as many as fit in 40 KiB and 64 (FP64) or 128 (FP32), keep all threads
// busy in stages of few butterflies.  Lengths of three stages have two exchange
// buffers and take narrow tiles only, which share a CU by three or more (two
// from 120 on in FP64).
constexpr int kNarrow = 16;
template <typename T2, int N>
constexpr int wide_tile() {
  int p = kNarrow;
  if (pencil_stages<T2>(N).nstage > 2) return p;
  while (2 * p * N * (int)sizeof(T2) <= 40960 && 2 * p * (int)sizeof(T2) <= 1024) p *= 2;
  return p;
}

// A pass takes wide tiles when they are 1.5 workgroups per CU or more and pad the
// pencils of a group by no more than 5 %, or by 1.5 or 2 times where a narrow tile's
// first stage is a quarter or an eighth of its threads.  Whole transforms, wide
// against narrow in both passes, us:  FP64 128 x 64^3 GTOR 207.5 against 216.7, one
// 72^3 19.6 against 17.7 (162 workgroups), 96 x 22^3 34.2 against 38.1 (first
// stages of two butterflies), 96 x 42^3 159 against 145 (three stages); FP32 12 x
// 64^3 38.9 against 41.8, one 80^3 26.1 against 18.0 (100 workgroups), 96 x 48^3
// 112.9 against 107.6 (48 pencils in tiles of 64), 96 x 36 x 36 x 12 (12 pencils
// in tiles of 128) 53 against 32.
constexpr int kWideMin = 384;
template <typename T2, int N>
bool use_wide(int npen, long groups) {
  constexpr int TP = wide_tile<T2, N>(), first = N / pencil_stages<T2>(N).radix[0];
  const long wide = (npen + TP - 1) / TP, narrow = (npen + kNarrow - 1) / kNarrow;
  const long limit = first <= 2 ? 200 : (first <= 4 ? 150 : 105);
  return 100 * wide * TP <= limit * narrow * kNarrow && wide * groups >= kWideMin;
}

// stage ST with the span NS = product of the earlier radices: the operations
// of the Stockham stages of pw_fft.hip.  One instance serves both signs, as
// there: the compiler folds the sign in after it has ordered the products and
// sums that it contracts, and an instance per sign rounds FP32 transforms
// differently from the run-time kernel's.
template <typename T2, int N, int TP, int ST, int NS>
__device__ inline void pencil_stage(const PencilIo<T2> &io, int q0, T2 *in, T2 *out, const T2 *__restrict__ tw,
                                    int sign) {
  constexpr Fft1D f = pencil_stages<T2>(N);
  constexpr int R = f.radix[ST], NBF = N / R, TWM = N / (NS * R);
  constexpr bool LAST = ST + 1 == f.nstage;
  for (int w = threadIdx.x; w < NBF * TP; w += kPB) {
    const int pen = w % TP, j = w / TP, k = j % NS;
    T2 v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if constexpr (ST == 0) v[r] = io.load(j + r * NBF, q0 + pen);
      else v[r] = in[(j + r * NBF) * TP + pen];
    }
    if constexpr (NS > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) {
        T2 t = tw[TWM * k * r];
        if (sign < 0) t.y = -t.y;
        v[r] = cmul(v[r], t);
      }
    }
    const int d = (j / NS) * NS * R + k;
    int row[R];
    if constexpr (LAST) {
#pragma unroll
      for (int r = 0; r < R; ++r) row[r] = io.out_row(d + r * NS);
    }
    dft<T2, R>(v, sign);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if constexpr (LAST) io.store(row[r], q0 + pen, v[r]);
      else out[(d + r * NS) * TP + pen] = v[r];
    }
  }
  if constexpr (!LAST) {
    __syncthreads();
    pencil_stage<T2, N, TP, ST + 1, NS * R>(io, q0, out, in, tw, sign);
  }
}

template <typename T2, int N, int TP, int SIGN, bool REAL>
__global__ void __launch_bounds__(kPB) k_pencil(PencilArgs a, const T2 *__restrict__ tw) {
  constexpr int NST = pencil_stages<T2>(N).nstage;
  // stage 0 writes b1; a third stage writes b0
  __shared__ T2 b1[NST > 1 ? N * TP : 1], b0[NST > 2 ? N * TP : 1];
  const int ntile = (a.npen + TP - 1) / TP, grp = blockIdx.x / ntile, q0 = (blockIdx.x - grp * ntile) * TP;
  const PencilIo<T2> io(a, grp, blockIdx.y, SIGN > 0, REAL);
  pencil_stage<T2, N, TP, 0, 1>(io, q0, b0, b1, tw, SIGN);
}

template <typename T2, int N, int TP>
void launch_tile(int sign, int nb, const PencilArgs &a, const void *tw, hipStream_t s) {
  const dim3 grid((unsigned)((a.npen + TP - 1) / TP * a.ngrp), nb);
  if constexpr (sizeof(T2) == sizeof(double2)) {
    if (a.real) {
      if (sign > 0) k_pencil<T2, N, TP, +1, true><<<grid, kPB, 0, s>>>(a, (const T2 *)tw);
      else k_pencil<T2, N, TP, -1, true><<<grid, kPB, 0, s>>>(a, (const T2 *)tw);
      return;
    }
  }
  if (sign > 0) k_pencil<T2, N, TP, +1, false><<<grid, kPB, 0, s>>>(a, (const T2 *)tw);
  else k_pencil<T2, N, TP, -1, false><<<grid, kPB, 0, s>>>(a, (const T2 *)tw);
}

template <typename T2, int N>
void launch(int sign, int nb, const PencilArgs &a, const void *tw, hipStream_t s) {
  constexpr int TP = wide_tile<T2, N>();
  if (TP > kNarrow && use_wide<T2, N>(a.npen, (long)a.ngrp * nb)) launch_tile<T2, N, TP>(sign, nb, a, tw, s);
  else launch_tile<T2, N, kNarrow>(sign, nb, a, tw, s);
}

}  // namespace

// the grid rule's lengths up to 144 (2^h 3^i 5^j 7^k 11^m, i <= 2, j, k, m <= 1,
// without those that carry both 7 and 11, or 5 and 11)
bool pencil_pass(const Fft1D &f, bool fp64, int sign, int nb, const PencilArgs &a, const void *tw, hipStream_t s) {
  switch (f.n) {
#define PW_N(N)                                                \
  case N:                                                      \
    if (fp64) launch<double2, N>(sign, nb, a, tw, s);          \
    else launch<float2, N>(sign, nb, a, tw, s);                \
    return true;
    PW_N(12) PW_N(14) PW_N(16) PW_N(18) PW_N(20) PW_N(22) PW_N(24) PW_N(28) PW_N(30) PW_N(32) PW_N(36) PW_N(40)
    PW_N(42) PW_N(44) PW_N(48) PW_N(56) PW_N(60) PW_N(64) PW_N(66) PW_N(70) PW_N(72) PW_N(80) PW_N(84) PW_N(88)
    PW_N(90) PW_N(96) PW_N(112) PW_N(120) PW_N(126) PW_N(128) PW_N(132) PW_N(140) PW_N(144)
#undef PW_N
    default: return false;
  }
}
