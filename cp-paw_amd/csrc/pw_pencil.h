// One pass of 1D transforms over pencils: the y and z passes of the full-grid
// PLANEWAVE$FFT.
#pragma once
#include "pw_common.h"

// Element e of pencil q sits at base + row stride + q in both arrays; row = e,
// but map[e] in the source of a forward (+1) pass and in the destination of an
// inverse pass (negative: reads as zero, is not written).  Bands and pencil
// groups are offset in both arrays; with grow the map of a group starts at
// nmap grow[group].
struct PencilArgs {
  const void *src;
  void *dst;
  int npen, ngrp;              // pencils of a group, groups
  const int *map, *grow;
  int nmap, sstride, dstride;
  bool real;                   // FP64: the grid side is a real array (imaginary parts zero / dropped)
  size_t sband, sgrp, dband, dgrp;
};

// src and dst of one (group, band).  A forward pass reads through its map, an
// inverse pass writes through it.  Loads are branch-free (an absent row or
// pencil reads a valid element and takes zero), so that the R loads of a
// butterfly go out together.
template <typename T2> struct PencilIo {
  const T2 *src;
  T2 *dst;
  const int *map;
  unsigned ss, ds;
  int npen;
  bool forward, real;   // constants in every kernel
  __device__ PencilIo(const PencilArgs &a, int grp, int band, bool forward, bool real)
      : src((const T2 *)a.src + band * a.sband + grp * a.sgrp), dst((T2 *)a.dst + band * a.dband + grp * a.dgrp),
        map(a.map + (a.grow ? a.nmap * a.grow[grp] : 0)), ss(a.sstride), ds(a.dstride), npen(a.npen),
        forward(forward), real(real) {
    // the real side counts elements of half the size (one group)
    if (real && forward) dst = (T2 *)((decltype(T2::x) *)a.dst + band * a.dband);
    if (real && !forward) src = (const T2 *)((const decltype(T2::x) *)a.src + band * a.sband);
  }
  __device__ T2 load(int e, int q) const {
    const int m = forward ? map[e] : e;
    const unsigned o = (unsigned)max(m, 0) * ss + (unsigned)min(q, npen - 1);
    T2 v;
    if (real && !forward) {
      v.x = reinterpret_cast<const decltype(v.x) *>(src)[o];
      v.y = 0;
    } else {
      v = src[o];
    }
    const bool ok = m >= 0 && q < npen;
    T2 z;
    z.x = ok ? v.x : 0;
    z.y = ok ? v.y : 0;
    return z;
  }
  // row of element e in dst, negative: not written.  Read before the first
  // store of a butterfly: a load behind a store waits for its own round trip
  __device__ int out_row(int e) const { return forward ? e : map[e]; }
  // streaming stores: a pass writes each element once and more than L2 holds
  __device__ void store(int m, int q, T2 v) const {
    typedef decltype(v.x) V2 __attribute__((ext_vector_type(2)));
    if (m < 0 || q >= npen) return;
    const unsigned i = (unsigned)m * ds + (unsigned)q;
    if (real && forward) {
      reinterpret_cast<decltype(v.x) *>(dst)[i] = v.x;
    } else {
      const V2 o = {v.x, v.y};
      __builtin_nontemporal_store(o, reinterpret_cast<V2 *>(dst + i));
    }
  }
};

// the pass by a kernel of the length fixed at compile time, false when the
// length has none; sign +1 or -1, tw = exp(+2 pi i m / n), m < n
bool pencil_pass(const Fft1D &f, bool fp64, int sign, int nb, const PencilArgs &a, const void *tw, hipStream_t s);
