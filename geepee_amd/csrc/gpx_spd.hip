// Batched SPD inverse + log-determinant: one workgroup per M x M matrix, or many for a few large
// ones.
//
// Replaces the per-output-dim np.linalg.inv / slogdet / solve calls of the layer
// algebra (base_models.py:462-476; aep_models.py:62-95, 523-533).  The matrix stays in
// registers, as MFMA accumulator tiles, for the whole inversion.
//
// Algorithm: Gauss-Jordan elimination without pivoting (stable for SPD input) over
// 16 x 16 pivot blocks, on the FP64 matrix cores (spd_gj_kernel below).
#include "gpx_common.h"

#include <utility>

namespace {

// LDS of one matrix.  Tiles are kept as the registers of the MFMA accumulator layout:
// [r][lane] with lane = 16 (row % 4) + column, row = 4r + lane / 16.
//   rv: block row K, one 256-double slot per tile J, the identity in slot K and the pivot
//       block P in slot MT; the panel replaces slot J by P^-1 A[K,J] and slot K by P^-1.
//       Register r of a slot is at the same time the k-slice r of an MFMA B operand.
//   ct: minus block column K transposed, [k][row] with rows of 17, per tile I (the MFMA A
//       operand of the updates); slot K holds the identity.
// With those identities and the tiles of block row and column K zeroed where they are
// published, every tile's update is the same A[I,J] += ct[I] rv[J], without a branch.
// Both double-buffered by the parity of K, so a wave may publish block K + 1 while others
// still update with block K; NB = 1 (one more barrier per block) where two do not fit.
// From M = 193 on the matrix and the working registers outgrow the register file: TL tiles per
// wave live in lt and, from M = 225 on, TG tiles at their place in the output array (in the
// L2), read and written once per block.  GT = false: no output array (log det only), those
// tiles in registers that spill.
template <int MT, int NW, bool GT>
struct SpdShape {
  static constexpr int T = MT * MT;
  static constexpr int TPW = (T + NW - 1) / NW;                 // tiles per wave
  static constexpr int TL = MT <= 12 ? 0 : (MT == 13 ? 1 : 5);  // of them in LDS
  static constexpr int TG = !GT || MT < 15 ? 0 : (MT == 15 ? 4 : 7);  // in the output array
  static constexpr int TR = TPW - TL - TG;                      // in registers
  static constexpr int NB = MT <= 13 ? 2 : 1;
  static constexpr int NPW = NW == 4 ? 3 : 6;  // waves that carry the panel's tiles
  static constexpr int NJ = (MT + NPW - 1) / NPW;               // tiles of each
  // where the accumulators leave few registers: the panel's tiles stay in LDS (YL), and the
  // updates load one tile's operands at a time (not PF)
  static constexpr bool YL = MT >= 13, PF = GT || MT <= 14;
};

template <int MT, int NW>
struct SpdLds {
  typedef SpdShape<MT, NW, true> S;
  static constexpr int CT = 16 * 17, COLS = MT, WAVES = NW, NPW = S::NPW, NJ = S::NJ;
  static constexpr bool YL = S::YL;
  // the small arrays first: LDS addresses below 64 KB fit an instruction's offset field
  double mul[4][16];   // [g][i]: pivot g's multiplier of row i, its reciprocal at i = g
  double piv[16 * MT];
  double red[16];
  int first[NW];
  int step;            // pivots done, in fours, over all blocks
  double pt[4][CT];    // the pivot block, transposed, before each four pivots
  double rv[S::NB][(MT + 1) * 256];
  double ct[S::NB][MT * CT];
  double lt[S::TL ? S::TL * NW * 256 : 1];
};

// Lane LC of each 16-lane row to the whole row (DPP row_newbcast, one instruction).
template <int LC>
__device__ __forceinline__ double spd_bcast16(double v) {
  return __longlong_as_double(
      __builtin_amdgcn_mov_dpp((long long)__double_as_longlong(v), 0x150 + LC, 0xF, 0xF, true));
}

// c[g][i] = the value of v in lane 4 g + i of each row.
template <int... E>
__device__ __forceinline__ void spd_spread(double v, double (*c)[4], std::integer_sequence<int, E...>) {
  ((c[E / 4][E % 4] = spd_bcast16<E>(v)), ...);
}

// x[k] = the value of v in lane 16 k + (lane % 16): the four 16-lane rows of v, each in
// every row (cross-row lane swaps).
__device__ __forceinline__ void spd_rows4(double v, double *x) {
  const unsigned lo = __double2loint(v), hi = __double2hiint(v);
  const auto l16 = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h16 = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
#pragma unroll
  for (int o = 0; o < 2; ++o) {  // o = 0: rows 0 and 2, o = 1: rows 1 and 3
    const auto l32 = __builtin_amdgcn_permlane32_swap(l16[o], l16[o], false, false);
    const auto h32 = __builtin_amdgcn_permlane32_swap(h16[o], h16[o], false, false);
    x[o] = __hiloint2double(h32[0], l32[0]);
    x[o + 2] = __hiloint2double(h32[1], l32[1]);
  }
}

__device__ __forceinline__ void spd_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 1/d from the hardware estimate r (relative error e < 2^-20): r (1 + e + e^2), three dependent
// operations after the estimate.
__device__ __forceinline__ double spd_recip(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// One scalar pivot, row 4 R + G of the pivot block, on the four rows x of its register R
// (each lane its column); c[G] the pivot's reciprocal, c[i] its multiplier of row i.
template <int R, int G>
__device__ __forceinline__ void spd_pivot(double *x, double *c, double &d) {
  d = spd_bcast16<4 * R + G>(x[G]);
  c[G] = spd_recip(d);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i != G) c[i] = spd_bcast16<4 * R + G>(x[i]);
  x[G] *= c[G];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i != G) x[i] = fma(-c[i], x[G], x[i]);
}

// x0 .. x3 by the lane's 16-lane row.
__device__ __forceinline__ double spd_pick(double x0, double x1, double x2, double x3, int lr) {
  const bool odd = lr & 1, high = lr & 2;
  return high ? (odd ? x3 : x2) : (odd ? x1 : x0);
}

// Rows 4R .. 4R+3 of the pivot block P (wave 0): four scalar pivots over the four rows, their
// multipliers to LDS for the other waves, then the rank-4 update of P's other rows as one
// MFMA.
template <int R, class L>
__device__ __forceinline__ void spd_pivot_rows(L &sm, int K, int lane, gpx_d4 &P) {
  const int lr = lane >> 4, lc = lane & 15;
  double x[4], c[4][4], d[4];
  spd_rows4(P[R], x);
  spd_pivot<R, 0>(x, c[0], d[0]);
  __builtin_amdgcn_sched_barrier(0);
  // A operand P[., 4R .. 4R+3] before these pivots (columns to operand layout through LDS)
#pragma unroll
  for (int r = 0; r < 4; ++r) sm.pt[R][lc * 17 + lr + 4 * r] = P[r];
  spd_wave_sync();
  const double a = sm.pt[R][(4 * R + lr) * 17 + lc];
  __builtin_amdgcn_sched_barrier(0);
  spd_pivot<R, 1>(x, c[1], d[1]);
  spd_pivot<R, 2>(x, c[2], d[2]);
  spd_pivot<R, 3>(x, c[3], d[3]);
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sm.mul[R][g * 4 + i] = c[g][i];
      sm.piv[K * 16 + 4 * R + g] = d[g];
    }
  }
  if constexpr (R < 3) {
    const double px = spd_pick(x[0], x[1], x[2], x[3], lr);
    P = gpx_mfma16(a, -px, P);
    P[R] = px;
  }
  __hip_atomic_store(&sm.step, 4 * K + R + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The same rows of the wave's panel tiles, one step behind the pivot block.
template <int R, class L>
__device__ __forceinline__ void spd_tile_rows(L &sm, double *rv, int K, int pw, int lane, gpx_d4 *y) {
  constexpr int MT = L::COLS, NJ = L::NJ;
  const int lr = lane >> 4, lc = lane & 15;
  // tile j of the wave; past the last tile the first one again (its copy is not written back)
  auto slot = [&](int j) { return rv + (pw + L::NPW * j < MT ? pw + L::NPW * j : pw) * 256; };
  double yr[NJ][4];
  if constexpr (R > 0 && !L::YL) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) slot(j)[R * 64 + lane] = y[j][R];
  }
  spd_wave_sync();
  auto rows = [&](int j) {
#pragma unroll
    for (int k = 0; k < 4; ++k) yr[j][k] = slot(j)[R * 64 + 16 * k + lc];
  };
  if constexpr (!L::YL) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) rows(j);
  }
  while (__hip_atomic_load(&sm.step, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < 4 * K + R + 1) {
    __builtin_amdgcn_s_sleep(1);  // leave instruction fetch to wave 0
  }
  const double a = sm.pt[R][(4 * R + lr) * 17 + lc];
  // the 16 multipliers as one value per lane of each row
  const double cm = sm.mul[R][lc];
  double c[4][4];
  spd_spread(cm, c, std::make_integer_sequence<int, 16>());
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if constexpr (L::YL) {
      if (pw + L::NPW * j >= MT) break;  // wave-uniform
      rows(j);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[j][r] = slot(j)[r * 64 + lane];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      yr[j][g] *= c[g][g];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i != g) yr[j][i] = fma(-c[g][i], yr[j][g], yr[j][i]);
    }
    const double py = spd_pick(yr[j][0], yr[j][1], yr[j][2], yr[j][3], lr);
    y[j] = gpx_mfma16(a, -py, y[j]);
    y[j][R] = py;
    if constexpr (L::YL) {
#pragma unroll
      for (int r = 0; r < 4; ++r) slot(j)[r * 64 + lane] = y[j][r];
    }
  }
}

// Phase 2 for block K: Gauss-Jordan over the 16 scalar pivots of P on [P | I | A[K, other
// columns]].  Wave 0 runs the pivots on P alone; the waves of the other SIMDs (not wave 4,
// which shares wave 0's) carry the tiles of the block row, each a step of four pivots
// behind it (sm.step; wave 0 waits for nobody, so every wait ends).
template <class L>
__device__ __forceinline__ void spd_panel(L &sm, double *rv, int K, int w, int lane) {
  constexpr int MT = L::COLS, NJ = L::NJ;
  if (w == 0) {
    __builtin_amdgcn_s_setprio(3);
    gpx_d4 P;
#pragma unroll
    for (int r = 0; r < 4; ++r) P[r] = rv[MT * 256 + r * 64 + lane];
    spd_pivot_rows<0>(sm, K, lane, P);
    spd_pivot_rows<1>(sm, K, lane, P);
    spd_pivot_rows<2>(sm, K, lane, P);
    spd_pivot_rows<3>(sm, K, lane, P);
    __builtin_amdgcn_s_setprio(0);
    return;
  }
  const int pw = w < 4 ? w - 1 : w - 2;
  if (w == 4 || pw >= MT) return;
  gpx_d4 y[NJ];
  if constexpr (!L::YL) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int J = pw + L::NPW * j < MT ? pw + L::NPW * j : pw;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[j][r] = rv[J * 256 + r * 64 + lane];
    }
  }
  spd_tile_rows<0>(sm, rv, K, pw, lane, y);
  spd_tile_rows<1>(sm, rv, K, pw, lane, y);
  spd_tile_rows<2>(sm, rv, K, pw, lane, y);
  spd_tile_rows<3>(sm, rv, K, pw, lane, y);
  if constexpr (!L::YL) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (pw + L::NPW * j >= MT) break;
#pragma unroll
      for (int r = 0; r < 4; ++r) rv[(pw + L::NPW * j) * 256 + r * 64 + lane] = y[j][r];
    }
  }
}

// Phase 1 for one tile: block row K and (negated, transposed) block column KJ to LDS.
template <class L>
__device__ __forceinline__ void spd_publish(double *rv, double *ct, int K, int KJ, int I, int J, gpx_d4 &acc,
                                            int lane) {
  if (__builtin_expect(I != K && J != KJ, 1)) return;
  const int lr = lane >> 4, lc = lane & 15;
  double *c = ct + I * L::CT + lc * 17 + lr;
  if (I == K) {
    double *v = rv + (J == KJ ? L::COLS : J) * 256 + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r * 64] = acc[r];
    if (J == KJ) {
#pragma unroll
      for (int r = 0; r < 4; ++r) c[4 * r] = rv[KJ * 256 + r * 64 + lane] = lr + 4 * r == lc ? 1.0 : 0.0;
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) c[4 * r] = -acc[r];
  }
  acc = gpx_d4{0.0, 0.0, 0.0, 0.0};
}

// The wave's next tile, NW further in row-major order (I = MT past the last one).
template <int MT, int NW>
__device__ __forceinline__ void spd_next(int &I, int &J) {
  J += NW % MT;
  I += NW / MT;
  if (J >= MT) {
    J -= MT;
    ++I;
  }
}

// log det and info from the pivots, thread k holding pivot k (1 past the last); returns info: the first pivot that is not a positive
// number, counted from 1 (0: none; what was computed after it is not used).
template <class L>
__device__ __forceinline__ int spd_finish(L &sm, double d, int b, double *logdet, int *info) {
  constexpr int NW = L::WAVES;
  static_assert(NW * 64 >= 16 * L::COLS, "one pivot per thread");
  const int k = threadIdx.x;
  const unsigned long long bad = __ballot(!(d > 0.0 && d < INFINITY));
  if ((k & 63) == 0) sm.first[k >> 6] = bad ? k + __ffsll(bad) : 0;
  const double ld = gpx_block_sum(log(d), sm.red);  // its barriers order sm.first
  int fail = 0;
#pragma unroll
  for (int w = NW - 1; w >= 0; --w) fail = sm.first[w] ? sm.first[w] : fail;
  if (k == 0) {
    if (logdet) logdet[b] = fail ? NAN : ld;
    if (info) info[b] = fail;
  }
  return fail;
}

// Blocked Gauss-Jordan on the matrix cores, 16 x 16 pivot blocks.  Eliminating block
// K with P = A[K,K] (rows of K: A[K,:], columns of K: c = A[:,K]):
//   A[I,J] -= c_I P^-1 A[K,J]     (I, J != K)
//   A[K,J] <- P^-1 A[K,J],  A[I,K] <- -c_I P^-1,  A[K,K] <- P^-1,
// and after every block the matrix holds A^-1.  All MT x MT tiles are kept, in MFMA
// accumulator layout, dealt round-robin to the waves: keeping only a symmetric half and
// mirroring it costs two orders of magnitude in accuracy downstream on ill-conditioned
// input, because the two halves of a computed inverse carry errors that cancel in later
// products.  Per block: (1) the owners of block row and column K publish them to LDS; (2)
// the panel waves run Gauss-Jordan over the 16 scalar pivots on [P | I | A[K, other
// columns]], giving P^-1 A[K,:] and P^-1 without ever multiplying by an explicit P^-1
// (which loses an order of magnitude on ill-conditioned blocks); (3) every wave updates
// its tiles with four 16x16x4 MFMAs per tile.  The scalar pivots are the D of A = L D L^T:
// their logs sum to log det A and the first non-positive one flags a matrix that is not
// positive definite.  The matrix is padded with the identity up to a multiple of 16.
//
// What bounds it: the serial chain of 16 pivots per block (about 3,900 cycles on wave 0; the
// tiles of the block row follow one step of four pivots behind, about 1,900 more) and the 4 T
// MFMAs of 64 cycles per block on four SIMDs (4,096 of them at M = 128, 10,816 at M = 200);
// an FP64 MFMA holds up the FP64 vector work of its SIMD, so the two do not overlap.  Every
// lane broadcast is a DPP move or a lane swap (16 rows of one column at a time by scalar
// lane reads took 6,700 cycles per block), and the updates run without a branch, the next
// tile's operands loaded beside the current MFMAs.  One matrix, microseconds before -> now:
// M = 50 18.3 -> 14.5, 100 43.5 -> 38, 128 53 -> 48, 160 102 -> 74, 200 200 -> 141,
// 224 255 -> 173, 256 409 -> 289 (64 matrices take 2-4% longer).
template <int MT, int NW, bool GT>
__global__ __launch_bounds__(NW * 64) void spd_gj_kernel(int M, int batch, const double *__restrict__ A,
                                                         int lda, long sA, double *__restrict__ out, int ldo,
                                                         long sO, double *__restrict__ logdet,
                                                         int *__restrict__ info) {
  typedef SpdShape<MT, NW, GT> S;
  constexpr int T = S::T, TR = S::TR, TL = S::TL, TG = S::TG, TM = TL + TG, CT = SpdLds<MT, NW>::CT;
  __shared__ SpdLds<MT, NW> sm;
  const int b = blockIdx.x;
  if (b >= batch) return;
  // w in a scalar register: the tile indices and their LDS offsets are then wave-uniform
  // scalars rather than a few vector registers per tile
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane >> 4, lc = lane & 15;
  const double *Ab = A + b * sA;
  gpx_d4 acc[TR];
  double *lt = sm.lt + (TL ? w * TL * 256 : 0);
  // tile t = w + NW u of the wave: u < TG in the output array (they lie in the first rows of
  // tiles, where the padding is the zeros right of column M), the next TL in LDS, the others
  // in acc.  Loads are unconditional at clamped indices (so they issue together); the identity padding of the
  // edge tiles is put in afterwards.
  auto load = [&](int t) {
    gpx_d4 v;
    const int I = t / MT, J = t % MT, j = min(J * 16 + lc, M - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = Ab[(long)min(I * 16 + lr + 4 * r, M - 1) * lda + j];
    return v;
  };
  auto pad = [&](int t, gpx_d4 &v) {
    const int I = t / MT, J = t % MT, j = J * 16 + lc;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = I * 16 + lr + 4 * r;
      v[r] = i < M && j < M ? v[r] : (i == j ? 1.0 : 0.0);
    }
  };
  double *Ob = out ? out + b * sO : nullptr;
  auto get = [&](int u, int I, int J) {
    gpx_d4 v;
    if (u < TG) {
      const int j = J * 16 + lc;
      const double *p = Ob + (long)(I * 16 + lr) * ldo + min(j, M - 1);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = p[(long)(4 * r) * ldo];
        if (j >= M) v[r] = 0.0;
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = lt[(u - TG) * 256 + r * 64 + lane];
    }
    return v;
  };
  auto put = [&](int u, int I, int J, const gpx_d4 &v) {
    if (u < TG) {
      const int j = J * 16 + lc;
      double *p = Ob + (long)(I * 16 + lr) * ldo + j;
      if (j < M) {
#pragma unroll
        for (int r = 0; r < 4; ++r) p[(long)(4 * r) * ldo] = v[r];
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) lt[(u - TG) * 256 + r * 64 + lane] = v[r];
    }
  };
  if (threadIdx.x == 0) sm.step = 0;
#pragma unroll
  for (int u = 0; u < TR; ++u) acc[u] = load(w + NW * (u + TM));
#pragma unroll
  for (int u = 0; u < TM; ++u) {
    gpx_d4 v = load(w + NW * u);
    if (M & 15) pad(w + NW * u, v);
    put(u, (w + NW * u) / MT, (w + NW * u) % MT, v);
  }
  if (M & 15) {  // wave-uniform
#pragma unroll
    for (int u = 0; u < TR; ++u) pad(w + NW * (u + TM), acc[u]);
  }
#pragma unroll 1
  for (int K = 0;; ++K) {
    const int buf = S::NB == 2 ? K & 1 : 0;
    double *rv = sm.rv[buf], *ct = sm.ct[buf];
    // the wave's first tile; opaque per block, so that the tile indices are stepped along
    // instead of being kept for every tile over the whole elimination
    int w0 = w;
    asm volatile("" : "+s"(w0));
    // (1) block row and column K to LDS
    {
      int I = w0 / MT, J = w0 % MT;
#pragma unroll
      for (int u = 0; u < TM + TR; ++u) {
        if (u < TM) {
          if (__builtin_expect(I == K || J == K, 0)) {
            gpx_d4 v = get(u, I, J);
            spd_publish<SpdLds<MT, NW>>(rv, ct, K, K, I, J, v, lane);
            put(u, I, J, v);
          }
        } else if (u + 1 < TM + TR || T % NW == 0 || I < MT) {
          spd_publish<SpdLds<MT, NW>>(rv, ct, K, K, I, J, acc[u < TM ? 0 : u - TM], lane);
        }
        spd_next<MT, NW>(I, J);
      }
    }
    __syncthreads();
    // (2) the panel
    spd_panel(sm, rv, K, w, lane);
    __syncthreads();
    // (3) the tiles, the next tile's operands loaded beside this one's MFMAs (hoisting more
    // of the LDS loads would hold all of them in registers at once); a wave's tile past the
    // last one is computed from the last row's operands and never used
    double a[2][4], bv[2][4];
    int I = w0 / MT, J = w0 % MT;
    auto operands = [&](double *av, double *bw) {
      const double *pr = rv + J * 256 + lane, *pc = ct + min(I, MT - 1) * CT + lr * 17 + lc;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        bw[ks] = pr[ks * 64];
        av[ks] = pc[ks * 68];
      }
    };
    if (S::PF) operands(a[0], bv[0]);
    gpx_d4 ahead = TG ? get(0, I, J) : gpx_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < TM + TR; ++u) {
      constexpr int N1 = S::PF ? 1 : 0;  // tiles loaded ahead
      const int Iu = I, Ju = J;
      gpx_d4 v = u < TG ? ahead : (u < TM ? get(u, I, J) : acc[u < TM ? 0 : u - TM]);
      if (N1 == 0 || u + 1 < TM + TR) {
        if (N1 || u > 0) spd_next<MT, NW>(I, J);
        operands(a[(u + N1) & 1], bv[(u + N1) & 1]);
        if (N1 && u + 1 < TG) ahead = get(u + 1, I, J);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) v = gpx_mfma16(a[u & 1][ks], bv[u & 1][ks], v);
      if (u < TM) put(u, Iu, Ju, v); else acc[u < TM ? 0 : u - TM] = v;
      __builtin_amdgcn_sched_barrier(0);
    }
    if (K + 1 == MT) break;
    if (S::NB == 1) __syncthreads();
  }
  const int fail = spd_finish(sm, (int)threadIdx.x < M ? sm.piv[threadIdx.x] : 1.0, b, logdet, info);
  if (!out) return;
  // the store indices are formed afresh from an opaque copy of the lane: otherwise the
  // compiler keeps the load's per-tile indices live through the whole elimination
  int lane2 = lane;
  asm volatile("" : "+v"(lane2));
  const int lr2 = lane2 >> 4, lc2 = lane2 & 15;
#pragma unroll
  for (int u = 0; u < TM + TR; ++u) {
    const int t = w + NW * u, I = t / MT, J = t % MT;
    if (t >= T || (u < TG && !fail)) continue;
    const gpx_d4 v = u < TM ? get(u, I, J) : acc[u < TM ? 0 : u - TM];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = I * 16 + lr2 + 4 * r, j = J * 16 + lc2;
      if (i < M && j < M) Ob[(long)i * ldo + j] = fail ? NAN : v[r];
    }
  }
}

template <int MT>
int launch_gj(int M, int batch, const double *A, int lda, long sA, double *out, int ldo, long sO,
                 double *logdet, int *info, hipStream_t st) {
  // 8 waves (two per SIMD) from M > 48 on: one wave's LDS operand loads hide behind the
  // other's MFMAs
  constexpr int NW = MT <= 3 ? 4 : 8;
  if (MT < 15 || out)
    hipLaunchKernelGGL((spd_gj_kernel<MT, NW, true>), dim3(batch), dim3(NW * 64), 0, st, M, batch, A, lda, sA, out,
                       ldo, sO, logdet, info);
  else
    hipLaunchKernelGGL((spd_gj_kernel<MT, NW, MT < 15>), dim3(batch), dim3(NW * 64), 0, st, M, batch, A, lda, sA,
                       out, ldo, sO, logdet, info);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

typedef int (*gj_fn)(int, int, const double *, int, long, double *, int, long, double *, int *, hipStream_t);
const gj_fn kGJ[16] = {launch_gj<1>,  launch_gj<2>,  launch_gj<3>,  launch_gj<4>,
                             launch_gj<5>,  launch_gj<6>,  launch_gj<7>,  launch_gj<8>,
                             launch_gj<9>,  launch_gj<10>, launch_gj<11>, launch_gj<12>,
                             launch_gj<13>, launch_gj<14>, launch_gj<15>, launch_gj<16>};

// ---------------------------------------------------------------------------
// The same elimination over many workgroups, four 16-blocks (one panel) at a time, two launches
// per panel:
//   spd_diag_kernel, one workgroup per matrix, runs the four blocks on the 64 x 64 diagonal block
//     alone and records the steps: per block the pivot rows' multipliers (mul), the columns before
//     each four pivots (aop), the columns c_I of the other three rows (cop) and the block row Wd;
//   spd_sweep_kernel, per column tile J and three row tiles, replays the recorded steps on the
//     panel's four tiles of column J (its last wave), which gives the block rows W_k[J] = P^-1 A[K,J] at
//     their own stage, forms c_k = A[I,K0+k] - sum_{l<k} c_l Wd_l[k] for its row tiles (a wave each)
//     and applies the four rank-16 updates.
// These are the operations of the one-workgroup kernel, tile for tile and in its order; no product
// with an explicit inverse of the 64 x 64 block, which would cost accuracy on ill-conditioned
// panels.  Bound by the diagonal blocks' pivot chains (14 us per panel) and the replay (9 us).
// Between panels the matrix lives in two scratch copies in tile order (a sweep reads one
// and writes the other), padded with the identity.
// ---------------------------------------------------------------------------
constexpr int SPD_NB = 4;     // 16-blocks per panel
constexpr int SPD_SWEEP = 3;  // row tiles of a sweep's workgroup, a wave each; its last wave replays

// Scratch of one matrix, in doubles.
struct SpdWork {
  static constexpr int MUL = 0, AOP = MUL + 4 * 64, COP = AOP + 4 * 256, REC = COP + 16 * 256;
  static constexpr int WD = REC, PIV = WD + 16 * 256, TMP = PIV + 256;
  static constexpr long size(int MT) { return TMP + 2L * MT * MT * 256; }
};

// A panel step's matrix before (src, first panel: the caller's) and after it.
struct SpdStep {
  const double *A;  // caller's matrix, first panel only
  int lda;
  long sA;
  double *out;  // caller's result, last panel only
  int ldo;
  long sO;
  double *work;
  int M, MT, K0, from, to;  // scratch copies read (-1: A) and written (-1: out)
};

__device__ __forceinline__ gpx_d4 spd_step_load(const SpdStep &p, int b, int I, int J, int lane) {
  const int lr = lane >> 4, j = J * 16 + (lane & 15);
  gpx_d4 v;
  if (p.from >= 0) {
    const double *t = p.work + b * SpdWork::size(p.MT) + SpdWork::TMP +
                      ((long)(p.from * p.MT + I) * p.MT + J) * 256 + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = t[r * 64];
  } else {
    const double *A = p.A + b * p.sA;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = I * 16 + lr + 4 * r;
      const double x = A[(long)min(i, p.M - 1) * p.lda + min(j, p.M - 1)];
      v[r] = i < p.M && j < p.M ? x : (i == j ? 1.0 : 0.0);
    }
  }
  return v;
}

__device__ __forceinline__ void spd_step_store(const SpdStep &p, int b, int I, int J, int lane, const gpx_d4 &v,
                                               bool fail) {
  const int lr = lane >> 4, j = J * 16 + (lane & 15);
  if (p.to >= 0) {
    double *t = p.work + b * SpdWork::size(p.MT) + SpdWork::TMP + ((long)(p.to * p.MT + I) * p.MT + J) * 256 + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r * 64] = v[r];
  } else {
    double *o = p.out + b * p.sO;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = I * 16 + lr + 4 * r;
      if (i < p.M && j < p.M) o[(long)i * p.ldo + j] = fail ? NAN : v[r];
    }
  }
}

struct SpdDiagLds {
  static constexpr int CT = 16 * 17, COLS = SPD_NB, WAVES = 8, NPW = 6, NJ = 1;
  static constexpr bool YL = false;
  double mul[4][16];
  double piv[16 * SPD_NB];
  double red[16];
  int first[WAVES];
  int step;
  double pt[4][CT];
  double rv[2][(SPD_NB + 1) * 256];
  double ct[2][SPD_NB * CT];
};

__global__ __launch_bounds__(512) void spd_diag_kernel(SpdStep p, double *__restrict__ logdet, int *__restrict__ info) {
  typedef SpdDiagLds L;
  constexpr int CT = L::CT, NB = SPD_NB;
  __shared__ L sm;
  const int b = blockIdx.x, nb = min(NB, p.MT - p.K0), tid = threadIdx.x;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane >> 4, lc = lane & 15;
  double *work = p.work + b * SpdWork::size(p.MT);
  // tiles (w / 4, w % 4) and two rows below; those past a last panel's nb blocks are the identity
  gpx_d4 acc[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int I = w / NB + 2 * u, J = w % NB;
    acc[u] = spd_step_load(p, b, p.K0 + min(I, nb - 1), p.K0 + min(J, nb - 1), lane);
    if (I >= nb || J >= nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[u][r] = I == J && lr + 4 * r == lc ? 1.0 : 0.0;
  }
  if (tid == 0) sm.step = 0;
#pragma unroll 1
  for (int K = 0; K < nb; ++K) {
    double *rv = sm.rv[K & 1], *ct = sm.ct[K & 1];
#pragma unroll
    for (int u = 0; u < 2; ++u) spd_publish<L>(rv, ct, K, K, w / NB + 2 * u, w % NB, acc[u], lane);
    __syncthreads();
    spd_panel(sm, rv, K, w, lane);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const double *pr = rv + (w % NB) * 256 + lane, *pc = ct + (w / NB + 2 * u) * CT + lr * 17 + lc;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) acc[u] = gpx_mfma16(pc[ks * 68], pr[ks * 64], acc[u]);
    }
    // the record of this block
    for (int e = tid; e < 1024; e += 512) {
      work[SpdWork::WD + K * 1024 + e] = rv[e];
      const int I = e >> 8, ks = (e >> 6) & 3, l = e & 63;
      work[SpdWork::COP + K * 1024 + e] = ct[I * CT + (l >> 4) * 17 + (l & 15) + ks * 68];
    }
    if (tid < 256) {
      const int R = tid >> 6;
      work[SpdWork::AOP + K * 256 + tid] = sm.pt[R][(4 * R + lr) * 17 + lc];
    }
    if (tid < 64) work[SpdWork::MUL + K * 64 + tid] = sm.mul[tid >> 4][tid & 15];
  }
  double *pivots = work + SpdWork::PIV;
  if (tid < 16 * nb) pivots[16 * p.K0 + tid] = sm.piv[tid];
  int fail = 0;
  if (p.to < 0) {  // the last panel: every pivot is known
    const double d = tid >= p.M ? 1.0 : (tid < 16 * p.K0 ? pivots[tid] : sm.piv[tid - 16 * p.K0]);
    fail = spd_finish(sm, d, b, logdet, info);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int I = w / NB + 2 * u, J = w % NB;
    if (I < nb && J < nb) spd_step_store(p, b, p.K0 + I, p.K0 + J, lane, acc[u], fail);
  }
}

struct SpdSweepLds {
  double rec[SpdWork::REC];
  double wl[SPD_NB][256];
  double ct[SPD_SWEEP][16 * 17];
};

__global__ __launch_bounds__(256) void spd_sweep_kernel(SpdStep p) {
  __shared__ SpdSweepLds sm;
  constexpr int NB = SPD_NB;
  const int J = blockIdx.x, b = blockIdx.z, nb = min(NB, p.MT - p.K0), tid = threadIdx.x;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane >> 4, lc = lane & 15;
  const int own = J >= p.K0 && J < p.K0 + nb ? J - p.K0 : -1;  // the panel's own columns
  const int row = blockIdx.y * SPD_SWEEP + w, I = row < p.K0 ? row : row + nb;
  const bool on = w < SPD_SWEEP && I < p.MT;
  const double *work = p.work + b * SpdWork::size(p.MT);
  // waves 0-2: their row's panel columns and its tile of column J; wave 3: the panel's tiles of
  // column J
  gpx_d4 c[NB], v = gpx_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int kk = p.K0 + min(k, nb - 1);
    c[k] = w < SPD_SWEEP ? spd_step_load(p, b, min(I, p.MT - 1), kk, lane) : spd_step_load(p, b, kk, J, lane);
  }
  if (own < 0 && w < SPD_SWEEP) v = spd_step_load(p, b, min(I, p.MT - 1), J, lane);
  double wd[NB][NB][4];  // waves 0-2: Wd_l[k], l < k; wave 3: wd[k][0] = Wd_k[own]
  if (w < SPD_SWEEP) {
#pragma unroll
    for (int k = 1; k < NB; ++k)
#pragma unroll
      for (int l = 0; l < k; ++l)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          wd[l][k][r] = work[SpdWork::WD + (min(l, nb - 1) * NB + min(k, nb - 1)) * 256 + r * 64 + lane];
  } else if (own >= 0) {
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) wd[k][0][r] = work[SpdWork::WD + (min(k, nb - 1) * NB + own) * 256 + r * 64 + lane];
  }
  if (own < 0) {  // 16 bytes a lane: REC is even, the scratch 16-byte aligned from its base
#pragma unroll
    for (int u = 0; u < (SpdWork::REC / 2 + 255) / 256; ++u) {
      const int e = min(tid + 256 * u, SpdWork::REC / 2 - 1);
      ((double2 *)sm.rec)[e] = ((const double2 *)work)[e];
    }
  }
  __syncthreads();
  double a[NB][4];
  if (w < SPD_SWEEP) {
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      if (k >= nb) break;
#pragma unroll
      for (int l = 0; l < k; ++l)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
          c[k] = gpx_mfma16(a[l][ks], wd[l][k][ks], c[k]);
      double *t = sm.ct[w];
      spd_wave_sync();
#pragma unroll
      for (int r = 0; r < 4; ++r) t[lc * 17 + lr + 4 * r] = -c[k][r];
      spd_wave_sync();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) a[k][ks] = t[lr * 17 + lc + ks * 68];
    }
  } else if (own >= 0) {
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sm.wl[k][r * 64 + lane] = wd[k][0][r];
  } else {
    double mul[NB][4], aop[NB][4];
#pragma unroll
    for (int K = 0; K < NB; ++K)
#pragma unroll
      for (int R = 0; R < 4; ++R) {
        mul[K][R] = sm.rec[SpdWork::MUL + K * 64 + R * 16 + lc];
        aop[K][R] = sm.rec[SpdWork::AOP + K * 256 + R * 64 + lane];
      }
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      if (K >= nb) break;
      gpx_d4 y = c[K];
#pragma unroll
      for (int R = 0; R < 4; ++R) {
        double yr[4], m[4][4];
        spd_rows4(y[R], yr);
        spd_spread(mul[K][R], m, std::make_integer_sequence<int, 16>());
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          yr[g] *= m[g][g];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (i != g) yr[i] = fma(-m[g][i], yr[g], yr[i]);
        }
        const double py = spd_pick(yr[0], yr[1], yr[2], yr[3], lr);
        y = gpx_mfma16(aop[K][R], -py, y);
        y[R] = py;
      }
      c[K] = y;
#pragma unroll
      for (int r = 0; r < 4; ++r) sm.wl[K][r * 64 + lane] = y[r];
#pragma unroll
      for (int d = 1; d < NB; ++d) {  // the next block's row first
        const int i = (K + d) % NB;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
          c[i] = gpx_mfma16(sm.rec[SpdWork::COP + (K * NB + i) * 256 + ks * 64 + lane], y[ks], c[i]);
      }
    }
  }
  bool fail = false;
  if (p.to < 0) {  // the last panel's launch knows every pivot
    for (int k = lane; k < p.M; k += 64) {
      const double d = work[SpdWork::PIV + k];
      fail |= !(d > 0.0 && d < INFINITY);
    }
    fail = __any(fail);
  }
  __syncthreads();
  if (w == SPD_SWEEP) {
    if (own < 0 && blockIdx.y == 0)
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (k < nb) spd_step_store(p, b, p.K0 + k, J, lane, c[k], fail);
    return;
  }
  if (!on) return;
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    if (k >= nb || k < own) continue;  // a column of the panel starts from zero at its stage
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) v = gpx_mfma16(a[k][ks], sm.wl[k][ks * 64 + lane], v);
  }
  spd_step_store(p, b, I, J, lane, v, fail);
}

int launch_split(int M, int batch, const double *A, int lda, long sA, double *out, int ldo, long sO, double *logdet,
                 int *info, double *work, hipStream_t st) {
  const int MT = (M + 15) / 16;
  SpdStep p = {A, lda, sA, out, ldo, sO, work, M, MT, 0, -1, -1};
  for (int t = 0; p.K0 < MT; ++t, p.K0 += SPD_NB) {
    const int nb = MT - p.K0 < SPD_NB ? MT - p.K0 : SPD_NB;
    p.from = t ? (t - 1) & 1 : -1;
    p.to = p.K0 + nb < MT ? t & 1 : -1;
    hipLaunchKernelGGL(spd_diag_kernel, dim3(batch), dim3(512), 0, st, p, logdet, info);
    GPX_CHECK_LAUNCH();
    hipLaunchKernelGGL(spd_sweep_kernel, dim3(MT, gpx_cdiv(MT - nb, SPD_SWEEP), batch), dim3(256), 0, st, p);
    GPX_CHECK_LAUNCH();
  }
  return GPX_OK;
}

// Whether the many-workgroup form is the faster one: it costs about 23 us per panel while its
// sweeps' workgroups fit the chip, the other 6 to 18 us per block on one CU per matrix.  us, 1 / 4 /
// 16 / 64 matrices, against one workgroup each: M = 144 60 / 60 / 70 / 116 : 59 / 59 / 60 / 62, 160
// 64 / 65 / 76 / 130 : 73 / 74 / 74 / 77, 176 69 / 70 / 91 / 167 : 89 / 90 / 91 / 93, 200 84 / 86 / 120 / 237 :
// 139 / 141 / 142 / 145, 256 96 / 99 / 155 / 382 : 288 / 289 / 291 / 298.
bool split_wins(int MT, int batch) {
  const long blocks = (long)batch * MT * gpx_cdiv(MT - SPD_NB, SPD_SWEEP);
  return MT >= 12 ? blocks <= 1024 : MT >= 10 && blocks <= 256;
}


// Pivot-failure flags of several SPD launches folded into one status word pair:
// status[0] = the largest info entry (0 = every matrix was positive definite),
// status[1] = max(status[1], status[0]) (sticky across evaluations until the host
// clears it).  One wave; the list descriptors travel by value in the kernel arguments,
// so a captured launch needs no host memory.
constexpr int kStatusLists = 16;
struct StatusLists {
  const int *ptr[kStatusLists];
  int count[kStatusLists];
};

__global__ void __launch_bounds__(64) status_fold_kernel(int nlists, StatusLists L, int *status) {
  int m = 0;
  for (int j = 0; j < nlists; ++j) {
    const int *p = L.ptr[j];
    for (int i = threadIdx.x; i < L.count[j]; i += 64) m = max(m, p[i]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  if (threadIdx.x == 0) {
    status[0] = m;
    status[1] = max(status[1], m);
  }
}

}  // namespace

extern "C" {

int gpx_status_fold(int nlists, const int *const *lists, const int *counts, int *status,
                    void *stream) {
  if (nlists < 0 || nlists > kStatusLists || !status || (nlists > 0 && (!lists || !counts)))
    return GPX_EINVAL;
  StatusLists L = {};
  for (int j = 0; j < nlists; ++j) {
    if (counts[j] < 0 || (counts[j] > 0 && !lists[j])) return GPX_EINVAL;
    L.ptr[j] = lists[j];
    L.count[j] = counts[j];
  }
  hipLaunchKernelGGL(status_fold_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, nlists, L, status);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// Largest M the SPD kit accepts.
int gpx_spd_max_m(void) { return 256; }

// For each b < batch: out[b] = inv(A[b]), logdet[b] = log det A[b], info[b] = 0, or
// info[b] = k+1 (and NaN outputs) when pivot k is not positive.  `out` may alias `A`
// (in-place) or be NULL (log-determinant only); logdet / info may be NULL.
int gpx_spd_inv_batched(int M, int batch, const double *A, int lda, long strideA, double *out,
                        int ldo, long strideOut, double *logdet, int *info, void *stream) {
  if (M < 0 || batch < 0 || M > 256) return GPX_EINVAL;
  if (M == 0 || batch == 0) return GPX_OK;
  if (!A || lda < M || (out && ldo < M)) return GPX_EINVAL;
  return kGJ[(M + 15) / 16 - 1](M, batch, A, lda, strideA, out, ldo, strideOut, logdet, info,
                                   (hipStream_t)stream);
}

// Scratch (doubles) of gpx_spd_inv_batched_ws; 0 where one workgroup per matrix is used anyway.
long gpx_spd_workspace(int M, int batch) {
  const int MT = (M + 15) / 16;
  return M < 1 || M > 256 || batch < 1 || !split_wins(MT, batch) ? 0 : batch * SpdWork::size(MT);
}

// gpx_spd_inv_batched with scratch (16-byte aligned; NULL, or out NULL: as without).
int gpx_spd_inv_batched_ws(int M, int batch, const double *A, int lda, long strideA, double *out, int ldo,
                           long strideOut, double *logdet, int *info, double *work, void *stream) {
  if (M < 0 || batch < 0 || M > 256) return GPX_EINVAL;
  if (!work || !out || gpx_spd_workspace(M, batch) == 0)
    return gpx_spd_inv_batched(M, batch, A, lda, strideA, out, ldo, strideOut, logdet, info, stream);
  if (!A || lda < M || ldo < M) return GPX_EINVAL;
  return launch_split(M, batch, A, lda, strideA, out, ldo, strideOut, logdet, info, work, (hipStream_t)stream);
}

}  // extern "C"
