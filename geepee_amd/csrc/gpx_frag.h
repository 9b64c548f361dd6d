// Matrix-core operands read straight from global memory.  K advances in groups of 8; of a group,
// lane group g = lane / 16 supplies k = 2 g + s to MFMA step s = 0, 1 (the same permutation of k
// in both operands), so an operand whose rows run along k is read as one 16-byte load per lane
// and one whose rows run across k as 128-byte row segments.
#pragma once
#include "gpx_common.h"

typedef double gpx_d2 __attribute__((ext_vector_type(2), aligned(8)));

template <int T>
struct GpxFrag {
  double v[2][T];
};

// Operand view of one wave: `p` is uniform (tile origin), `off[i]` the lane's offset in tile i.
// KC: k is the contiguous dimension (row stride ld); otherwise k-rows of stride ld.
template <int T, bool KC>
struct GpxOperand {
  const double *p;
  long off[T];
  int ld;
  __device__ __forceinline__ GpxOperand(const double *base, int ld_, int r0, int rows, int lane) : ld(ld_) {
    const int g = lane >> 4, last = rows - r0 - 1;
    p = KC ? base + (long)r0 * ld : base + r0;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const int r = min(16 * i + (lane & 15), last);
      off[i] = KC ? (long)r * ld + 2 * g : 2L * g * ld + r;
    }
  }
  __device__ __forceinline__ void load(GpxFrag<T> &f, int k0) const {
    const double *q = p + (KC ? (long)k0 : (long)k0 * ld);
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if constexpr (KC) {
        const gpx_d2 t = *(const gpx_d2 *)(q + off[i]);
        f.v[0][i] = t.x;
        f.v[1][i] = t.y;
      } else {
        f.v[0][i] = q[off[i]];
        f.v[1][i] = (q + ld)[off[i]];
      }
    }
  }
  // the `kr` (1..7) valid k of a last group; lanes past them re-read the group's first
  __device__ __forceinline__ void load_tail(GpxFrag<T> &f, int k0, int kr, int lane) const {
    const double *q = p + (KC ? (long)k0 : (long)k0 * ld);
    const int g = lane >> 4;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bool on = 2 * g + s < kr;
      const long back = on ? s : -2 * g;
#pragma unroll
      for (int i = 0; i < T; ++i) {
        f.v[s][i] = 0.0;
        if constexpr (T > 2) {  // no registers for the clamped addresses
          if (on) f.v[s][i] = q[off[i] + (KC ? s : (long)s * ld)];
        } else {
          const double t = q[off[i] + (KC ? back : back * ld)];
          if (on) f.v[s][i] = t;
        }
      }
    }
  }
};
