// psi statistics of the ARD SE kernel under Gaussian inputs and their adjoint.
//
// Forward: compute_psi_weave (kernels.py:181-240, loop :201-234)
//   psi1[n,m]   = sf2 prod_q (l/(l+v))^1/2 exp(-(mu-z_m)^2 / (2(l+v)))
//   psi2[n,a,b] = sf2^2 prod_q (l/(l+2v))^1/2
//                 exp(-(z_a-z_b)^2/(4l) - (mu-(z_a+z_b)/2)^2/(2v+l))
// with l = ell^2 = exp(2 ls) and sf2 = exp(2 sf).  psi2 is written exactly
// symmetric: every value is computed once and stored at (a,b) and (b,a).
//
// Adjoint: compute_psi_derivatives -> psi1compDer / psi2compDer (kernels.py:302-309,
// 355-444), restated with per-point sufficient statistics.  With
// L[n,a,b] = dpsi2[n,a,b] psi2[n,a,b], T_na = sum_b L_nab,
// V_nq = sum_ab L_nab z_aq z_bq, S0 = sum_a T_a, S1_q = sum_a T_a z_aq,
// S2_q = (sum_a T_a z_aq^2 + V_q)/2 and d = 1/(2v+l):
//   dmu = -2 d (mu S0 - S1),  dv = 2 d^2 (mu^2 S0 - 2 mu S1 + S2) - d S0,
//   dell (per n) = 2 ell [(v/l) d S0 + d^2 (mu^2 S0 - 2 mu S1 + S2)
//                         + (sum_a T_a z_aq^2 - V_q) / (2 l^2)],
//   dZ_aq = sum_n [(U_naq - z_aq T_na)/l + d (2 mu T_na - z_aq T_na - U_naq)],  U_n = L_n z.
// A dpsi2 that is not symmetric enters as its symmetric part.
#include "gpx_frag.h"

#define GPX_QMAX 16

namespace {

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------

// PSI1_PTS points per block: their constants (w = 1 / (2 (v + l)) per q, and
// lc = sum_q log(l / (l + v)) / 2) are formed once in LDS, then thread (point, m) sums
// its Q terms; a row of M entries is written contiguously.
constexpr int PSI1_PTS = 4;

__global__ __launch_bounds__(256) void psi1_kernel(int N, int M, int Q, const double *__restrict__ mx,
                                                    const double *__restrict__ vx,
                                                    const double *__restrict__ z,
                                                    const double *__restrict__ ls,
                                                    const double *__restrict__ sf,
                                                    double *__restrict__ psi1) {
  __shared__ double lam[GPX_QMAX], pw[PSI1_PTS][GPX_QMAX], pm[PSI1_PTS][GPX_QMAX], plc[PSI1_PTS];
  const int tid = threadIdx.x, n0 = blockIdx.x * PSI1_PTS;
  if (tid < Q) lam[tid] = exp(2.0 * ls[tid]);
  __syncthreads();
  if (tid < PSI1_PTS * Q) {
    const int pt = tid / Q, q = tid % Q, n = min(n0 + pt, N - 1);
    const double v = vx[(long)n * Q + q];
    pw[pt][q] = 1.0 / (2.0 * (v + lam[q]));
    pm[pt][q] = mx[(long)n * Q + q];
  }
  if (tid < PSI1_PTS) {
    const int n = min(n0 + tid, N - 1);
    double lc = 0.0;
    for (int q = 0; q < Q; ++q) lc += 0.5 * log(lam[q] / (lam[q] + vx[(long)n * Q + q]));
    plc[tid] = lc;
  }
  __syncthreads();
  const double sf2 = exp(2.0 * sf[0]);
  for (int e = tid; e < PSI1_PTS * M; e += 256) {
    const int pt = e / M, m = e % M, n = n0 + pt;
    if (n >= N) break;
    double acc = 0.0;
    for (int q = 0; q < Q; ++q) {
      const double d = pm[pt][q] - z[m * Q + q];
      acc -= d * d * pw[pt][q];
    }
    psi1[(long)n * M + m] = sf2 * exp(acc + plc[pt]);
  }
}

// One block per (32 x 32 tile pair ta >= tb, chunk of PSI2_CH points).  Wave w computes
// the 16 x 16 block (w >> 1, w & 1) of the tile for every point of the chunk, lane l the
// entries (row (l >> 4) + 4r, column l & 15), r < 4.  The per-pair terms zh_q = (z_aq +
// z_bq)/2 and P_ab = sum_q (z_aq - z_bq)^2 / (4 l_q) stay in registers across the points,
// the points' constants are formed once per block in LDS, and an off-diagonal tile's
// mirrored block goes out through a wave-private LDS transpose: after the set-up no wave
// waits for another, and every store writes 128-byte row segments.
// QC: compile-time bound on Q (register arrays).
constexpr int PSI2_CH = 16;

template <int QC>
__global__ __launch_bounds__(256) void psi2_kernel(int N, int M, int Q, const double *__restrict__ mx,
                                                    const double *__restrict__ vx,
                                                    const double *__restrict__ z,
                                                    const double *__restrict__ ls,
                                                    const double *__restrict__ sf,
                                                    double *__restrict__ psi1,
                                                    double *__restrict__ psi2) {
  __shared__ double pmu[PSI2_CH][QC], pdd[PSI2_CH][QC], plc[PSI2_CH];
  __shared__ double pw1[PSI2_CH][QC], plc1[PSI2_CH];  // psi1 constants (tile pair 0 only)
  __shared__ double lam[QC], i4l[QC];
  __shared__ double tr[4][16][17];
  int p = blockIdx.x, ta = 0;
  while (p > ta) { p -= ta + 1; ++ta; }
  const int tb = p;
  const int a0 = ta * 32, b0 = tb * 32, tid = threadIdx.x;
  const int n0 = blockIdx.y * PSI2_CH, nend = min(N, n0 + PSI2_CH);
  if (tid < Q) {
    const double l = exp(2.0 * ls[tid]);
    lam[tid] = l;
    i4l[tid] = 1.0 / (4.0 * l);
  }
  __syncthreads();
  // point constants: mu, d = 1/(2v + l) (zero beyond Q, so the loops below run to QC
  // without branches) and lc = sum_q log(l / (l + 2v)) / 2
  for (int e = tid; e < PSI2_CH * QC; e += 256) {
    const int pt = e / QC, q = e % QC, n = min(n0 + pt, N - 1);
    const bool in = q < Q;
    pmu[pt][q] = in ? mx[(long)n * Q + q] : 0.0;
    pdd[pt][q] = in ? 1.0 / (2.0 * vx[(long)n * Q + q] + lam[q]) : 0.0;
  }
  if (tid < PSI2_CH) {
    const int n = min(n0 + tid, N - 1);
    double lc = 0.0;
    for (int q = 0; q < Q; ++q) lc += 0.5 * log(lam[q] / (lam[q] + 2.0 * vx[(long)n * Q + q]));
    plc[tid] = lc;
  }
  // the blocks of tile pair 0 also write psi1 for their points (one launch for both)
  const bool do_psi1 = blockIdx.x == 0;
  if (do_psi1) {
    for (int e = tid; e < PSI2_CH * Q; e += 256) {
      const int pt = e / Q, q = e % Q, n = min(n0 + pt, N - 1);
      pw1[pt][q] = 1.0 / (2.0 * (vx[(long)n * Q + q] + lam[q]));
    }
    if (tid >= 64 && tid < 64 + PSI2_CH) {
      const int pt = tid - 64, n = min(n0 + pt, N - 1);
      double lc = 0.0;
      for (int q = 0; q < Q; ++q) lc += 0.5 * log(lam[q] / (lam[q] + vx[(long)n * Q + q]));
      plc1[pt] = lc;
    }
  }
  __syncthreads();
  const double sf2 = exp(2.0 * sf[0]), sf4 = sf2 * sf2;
  if (do_psi1) {
    for (int e = tid; e < PSI2_CH * M; e += 256) {
      const int pt = e / M, m = e % M, n = n0 + pt;
      if (n >= nend) break;
      double acc = 0.0;
      for (int q = 0; q < Q; ++q) {
        const double d = pmu[pt][q] - z[m * Q + q];
        acc -= d * d * pw1[pt][q];
      }
      psi1[(long)n * M + m] = sf2 * exp(acc + plc1[pt]);
    }
  }
  const int lane = tid & 63, w = tid >> 6;
  const int ra = (w >> 1) * 16 + (lane >> 4), cb = (w & 1) * 16 + (lane & 15);
  const int b = b0 + cb, bl = min(b, M - 1);
  double zh[4][QC], P[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int al = min(a0 + ra + 4 * r, M - 1);  // padding rows read a real z row; never stored
    double pp = 0.0;
#pragma unroll
    for (int q = 0; q < QC; ++q) {
      if (q < Q) {
        const double x = z[al * Q + q], y = z[bl * Q + q];
        const double dz = x - y;
        zh[r][q] = 0.5 * (x + y);
        pp += dz * dz * i4l[q];
      } else {
        zh[r][q] = 0.0;
      }
    }
    P[r] = pp;
  }
  const bool mirror = ta != tb;
  // mirrored block: lane l writes row b0 + (w & 1) * 16 + (l >> 4) + 4r, columns
  // a0 + (w >> 1) * 16 + (l & 15)
  const int mb = b0 + (w & 1) * 16 + (lane >> 4), ma = a0 + (w >> 1) * 16 + (lane & 15);
  for (int n = n0; n < nend; ++n) {
    const int pt = n - n0;
    const double lc = plc[pt];
    double *out = psi2 + (long)n * M * M;
    double val[4], m[QC], d[QC];
#pragma unroll
    for (int q = 0; q < QC; ++q) {
      m[q] = pmu[pt][q];
      d[q] = pdd[pt][q];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double e = lc - P[r];
#pragma unroll
      for (int q = 0; q < QC; ++q) {
        const double h = m[q] - zh[r][q];
        e -= h * h * d[q];
      }
      val[r] = sf4 * exp(e);
      const int a = a0 + ra + 4 * r;
      if (a < M && b < M) __builtin_nontemporal_store(val[r], out + (long)a * M + b);
    }
    if (mirror) {
#pragma unroll
      for (int r = 0; r < 4; ++r) tr[w][(lane >> 4) + 4 * r][lane & 15] = val[r];
      // the wave reads what its other lanes wrote: order the LDS accesses at wave scope
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int bb = mb + 4 * r;
        const double v = tr[w][lane & 15][(lane >> 4) + 4 * r];
        if (bb < M && ma < M) __builtin_nontemporal_store(v, out + (long)bb * M + ma);
      }
      // and before the next point overwrites the buffer
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

// ---------------------------------------------------------------------------
// adjoint, materialised psi2
// ---------------------------------------------------------------------------

// One workgroup per point, point after point.  With L = dpsi2_n * psi2_n the matrix cores form
// U = L z (as U^T = z^T L: L's elements are the B operand exactly as they are read, 128-byte row
// segments), T = the row sums of L ride along on the vector ALU, and everything the adjoint needs
// is linear in U, T and Lp = dpsi1 * psi1:
//   dZ_aq += (U - z T)/l + d (2 mu T - z T - U) + Lp e (mu - z),  d = 1/(2v+l), e = 1/(v+l),
// summed over the workgroup's points in registers (lane (g, c): q = g + 4 r, a = n0 + 16 j + c),
// and the per-point sums S0, S1, TZ2, V and the psi1 terms, reduced over a across the 16 lanes of
// a row and then over the waves.  The L array, its product with [1 | d] and the T, Lp products
// are not formed.  SYM: dpsi2 is symmetric; otherwise L uses (dpsi2 + dpsi2^T)/2, whose transposed
// reads come from the caches.  Bound by reading psi2 and dpsi2 once: N = 1501, M = 100, Q = 5 65 us
// (78 with the symmetric part taken here), 50 at the rate of a large copy; one thread per column,
// with L stored and its product, 260 + 66 (and 122 for a symmetrising pass).  N = 1000 134 -> 48.
// part[block]: [dZ (M x Q) | sum of H (Q) | S0, A1].
constexpr int PSI_NRED = 5 * GPX_QMAX + 2;
constexpr int PSI_ZLD = GPX_QMAX + 1;

template <int TN, int W, bool SYM>
__global__ __launch_bounds__(64 * W, 3) void psi_bwd_points_kernel(
    int N, int M, int Q, const double *__restrict__ mx, const double *__restrict__ vx,
    const double *__restrict__ z, const double *__restrict__ ls, const double *__restrict__ dpsi1,
    const double *__restrict__ psi1, const double *__restrict__ dpsi2, const double *__restrict__ psi2,
    double *__restrict__ dmx, double *__restrict__ dvx, double *__restrict__ part) {
  extern __shared__ double psi_lds[];
  const int Mp = (M + 7) & ~7, tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  double *zs = psi_lds;                                             // Mp x PSI_ZLD, zero padded
  double(*red)[W][PSI_NRED] = (double(*)[W][PSI_NRED])(zs + Mp * PSI_ZLD);  // [2][W][PSI_NRED]
  for (int e = tid; e < Mp * PSI_ZLD; e += 64 * W) {
    const int a = e / PSI_ZLD, q = e % PSI_ZLD;
    zs[e] = (a < M && q < Q) ? z[a * Q + q] : 0.0;
  }
  __syncthreads();
  const int nt = (M + 15) >> 4, lo = nt / W, hi = nt % W, tn = lo + (w < hi);
  const int first = 16 * (w * lo + min(w, hi)), n0 = min(first, M - 1);
  bool on[TN];
  double dz[TN][4];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    on[j] = j < tn && first + 16 * j + c < M;
#pragma unroll
    for (int r = 0; r < 4; ++r) dz[j][r] = 0.0;
  }
  double l[4], il[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    l[r] = g + 4 * r < Q ? exp(2.0 * ls[g + 4 * r]) : 1.0;
    il[r] = 1.0 / l[r];
  }
  const GpxOperand<TN, false> off(psi2, M, n0, M, lane);  // lane offsets of a point's matrix
  const GpxOperand<TN, true> offT(dpsi2, M, n0, M, lane);
  const int groups = M >> 3, kr = M & 7;
  const double *zl = zs + 2 * g * PSI_ZLD + c;  // A operand: z^T[q = c][k = 2 g + s]
  double hsum = 0.0, s0sum = 0.0, a1sum = 0.0;
  int par = 0;
  for (int n = blockIdx.x; n < N; n += gridDim.x, par ^= 1) {
    GpxOperand<TN, false> op = off, og = off;
    GpxOperand<TN, true> ot = offT;
    op.p = psi2 + (long)n * M * M + n0;
    og.p = dpsi2 + (long)n * M * M + n0;
    ot.p = dpsi2 + (long)n * M * M + (long)n0 * M;
    gpx_d4 U[TN];
    double T[TN], Lp[TN], p1[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      U[j] = gpx_d4{0.0, 0.0, 0.0, 0.0};
      T[j] = 0.0;
      const long e = (long)n * M + min(first + 16 * j + c, M - 1);
      Lp[j] = dpsi1[e];
      p1[j] = psi1[e];
    }
    GpxFrag<TN> fp[2], fg[2], ft[2];
    auto load = [&](int u, int t) {
      const int k0 = 8 * min(t, groups - 1);
      op.load(fp[u], k0);
      og.load(fg[u], k0);
      if constexpr (!SYM) ot.load(ft[u], k0);
    };
    auto mul = [&](int u, int t) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const double za = zl[(8 * t + s) * PSI_ZLD];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const double gg = SYM ? fg[u].v[s][j] : 0.5 * (fg[u].v[s][j] + ft[u].v[s][j]);
          const double le = gg * fp[u].v[s][j];
          T[j] += le;
          U[j] = gpx_mfma16(za, le, U[j]);
        }
      }
    };
    if (groups) {
      load(0, 0);
      int t = 0;
      for (; t + 2 <= groups; t += 2) {
        load(1, t + 1);
        mul(0, t);
        load(0, t + 2);
        mul(1, t + 1);
      }
      if (t < groups) mul(0, t);
    }
    if (kr) {
      op.load_tail(fp[0], 8 * groups, kr, lane);
      og.load_tail(fg[0], 8 * groups, kr, lane);
      if constexpr (!SYM) ot.load_tail(ft[0], 8 * groups, kr, lane);
      mul(0, groups);
    }
    double S0 = 0.0, A1 = 0.0;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      T[j] = on[j] ? gpx_swap_add<16>(gpx_swap_add<32>(T[j])) : 0.0;
      Lp[j] = on[j] ? Lp[j] * p1[j] : 0.0;
      S0 += T[j];
      A1 += Lp[j];
    }
    double *rw = red[par][w];
    int zo = first + c;  // opaque: z is re-read from LDS for each point, not kept in registers
    asm volatile("" : "+v"(zo));
    S0 = gpx_row_sum(S0);
    A1 = gpx_row_sum(A1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (4 * r >= Q) break;
      const int q = g + 4 * r, qc = min(q, Q - 1);
      const double mu = mx[(long)n * Q + qc], vv = vx[(long)n * Q + qc];
      const double d = 1.0 / (2.0 * vv + l[r]), e = 1.0 / (vv + l[r]);
      double V = 0.0, S1 = 0.0, Z2 = 0.0, B1 = 0.0, C1 = 0.0;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const double u = on[j] ? U[j][r] : 0.0, zz = zs[min(zo + 16 * j, M - 1) * PSI_ZLD + q];
        const double zm = zz - mu, tz = T[j] * zz, lz = Lp[j] * zm;
        V = fma(u, zz, V);
        S1 += tz;
        Z2 = fma(tz, zz, Z2);
        B1 += lz;
        C1 = fma(lz, zm, C1);
        dz[j][r] += fma(u - tz, il[r], d * (2.0 * mu * T[j] - tz - u)) - e * lz;
      }
      V = gpx_row_sum(V);
      S1 = gpx_row_sum(S1);
      Z2 = gpx_row_sum(Z2);
      B1 = gpx_row_sum(B1);
      C1 = gpx_row_sum(C1);
      if (c == 0) {
        rw[2 + q] = S1;
        rw[2 + GPX_QMAX + q] = Z2;
        rw[2 + 2 * GPX_QMAX + q] = V;
        rw[2 + 3 * GPX_QMAX + q] = B1;
        rw[2 + 4 * GPX_QMAX + q] = C1;
      }
    }
    if (lane == 0) {
      rw[0] = S0;
      rw[1] = A1;
    }
    __syncthreads();  // red[par] is next written two points on, behind the next point's barrier
    if (tid < Q) {
      const int q = tid;
      auto sum = [&](int i) {
        double t = red[par][0][i];
        for (int u = 1; u < W; ++u) t += red[par][u][i];
        return t;
      };
      const double s0 = sum(0), a1 = sum(1), s1 = sum(2 + q), tz2 = sum(2 + GPX_QMAX + q),
                   vs = sum(2 + 2 * GPX_QMAX + q), b1 = sum(2 + 3 * GPX_QMAX + q), c1 = sum(2 + 4 * GPX_QMAX + q);
      const double m = mx[(long)n * Q + q], v = vx[(long)n * Q + q];
      const double ell = exp(ls[q]), lq = exp(2.0 * ls[q]);
      const double d = 1.0 / (2.0 * v + lq), e = 1.0 / (v + lq);
      const double quad = m * m * s0 - 2.0 * m * s1 + 0.5 * (tz2 + vs);
      dmx[(long)n * Q + q] = -2.0 * d * (m * s0 - s1) + e * b1;
      dvx[(long)n * Q + q] = 2.0 * d * d * quad - d * s0 + 0.5 * e * (e * c1 - a1);
      hsum += 2.0 * ell * ((v / lq) * d * s0 + d * d * quad + (tz2 - vs) / (2.0 * lq * lq));
      hsum += e * ell * (e * c1 + (v / lq) * a1);
      s0sum += s0;
      a1sum += a1;
    }
  }
  double *po = part + (long)blockIdx.x * (M * Q + Q + 2);
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (on[j] && g + 4 * r < Q) po[(first + 16 * j + c) * Q + g + 4 * r] = dz[j][r];
  if (tid < Q) po[M * Q + tid] = hsum;
  if (tid == 0) {
    po[M * Q + Q] = s0sum;
    po[M * Q + Q + 1] = a1sum;
  }
}

// Sums the workgroups' partials (fixed order: 8 interleaved groups, then the groups).  A workgroup
// takes 32 of the M Q + Q + 1 outputs; the last output is dsf2 = (A1 + 2 S0) / sf2.
__global__ __launch_bounds__(256) void psi_bwd_sum_kernel(int M, int Q, int blocks, const double *__restrict__ part,
                                                          const double *__restrict__ sf, double *__restrict__ dsf2,
                                                          double *__restrict__ dell, double *__restrict__ dZ) {
  __shared__ double red[8][33];
  const int o = threadIdx.x & 31, g = threadIdx.x >> 5, mq = M * Q, width = mq + Q + 2;
  const int e = blockIdx.x * 32 + o;
  double s = 0.0;
  if (e < mq + Q) {
#pragma unroll 4
    for (int b = g; b < blocks; b += 8) s += part[(long)b * width + e];
  } else if (e == mq + Q) {
#pragma unroll 4
    for (int b = g; b < blocks; b += 8) s += part[(long)b * width + e + 1] + 2.0 * part[(long)b * width + e];
  }
  red[g][o] = s;
  __syncthreads();
  if (g != 0 || e > mq + Q) return;
  double t = red[0][o];
#pragma unroll
  for (int h = 1; h < 8; ++h) t += red[h][o];
  if (e < mq) dZ[e] = t;
  else if (e < mq + Q) dell[e - mq] = t;
  else dsf2[0] = t / exp(2.0 * sf[0]);
}

// Workgroups of the point pass: what fills three waves per SIMD, each with as many points as the
// others.
int psi_bwd_blocks(int N, int M) {
  const int most = M > 128 ? 256 : 768, rounds = (int)gpx_cdiv(N, most);
  return (int)gpx_cdiv(N, rounds);
}

template <int TN, int W>
int psi_bwd_launch(int blocks, int N, int M, int Q, int sym, const double *mx, const double *vx, const double *z,
                   const double *ls, const double *dpsi1, const double *psi1, const double *dpsi2,
                   const double *psi2, double *dmx, double *dvx, double *part, hipStream_t st) {
  const int lds = (int)sizeof(double) * (((M + 7) & ~7) * PSI_ZLD + 2 * W * PSI_NRED);
  if (sym)
    hipLaunchKernelGGL((psi_bwd_points_kernel<TN, W, true>), dim3(blocks), dim3(64 * W), lds, st, N, M, Q, mx, vx, z,
                       ls, dpsi1, psi1, dpsi2, psi2, dmx, dvx, part);
  else
    hipLaunchKernelGGL((psi_bwd_points_kernel<TN, W, false>), dim3(blocks), dim3(64 * W), lds, st, N, M, Q, mx, vx, z,
                       ls, dpsi1, psi1, dpsi2, psi2, dmx, dvx, part);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

}  // namespace

extern "C" {

int gpx_psi_qmax(void) { return GPX_QMAX; }

// psi1 (N x M) and, if psi2 != NULL, psi2 (N x M x M) for inputs x_n ~ N(mx_n, diag vx_n).
// ls (Q) and sf (1) are the raw log hyper-parameters on the device.
int gpx_psi_fwd(int N, int M, int Q, const double *mx, const double *vx, const double *z,
                const double *ls, const double *sf, double *psi1, double *psi2, void *stream) {
  if (N < 0 || M < 0 || Q < 1 || Q > GPX_QMAX) return GPX_EINVAL;
  if (N == 0 || M == 0) return GPX_OK;
  if (!mx || !vx || !z || !ls || !sf || !psi1) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (!psi2) {
    hipLaunchKernelGGL(psi1_kernel, dim3(gpx_cdiv(N, PSI1_PTS)), dim3(256), 0, st, N, M, Q, mx, vx, z, ls, sf,
                       psi1);
    GPX_CHECK_LAUNCH();
  } else {
    const int T = (M + 31) / 32;
    const unsigned chunks = gpx_cdiv(N, PSI2_CH);
    if (chunks > 65535) return GPX_EINVAL;
    const dim3 grid(T * (T + 1) / 2, chunks);
    if (Q <= 4)
      hipLaunchKernelGGL(psi2_kernel<4>, grid, dim3(256), 0, st, N, M, Q, mx, vx, z, ls, sf, psi1, psi2);
    else if (Q <= 8)
      hipLaunchKernelGGL(psi2_kernel<8>, grid, dim3(256), 0, st, N, M, Q, mx, vx, z, ls, sf, psi1, psi2);
    else
      hipLaunchKernelGGL(psi2_kernel<GPX_QMAX>, grid, dim3(256), 0, st, N, M, Q, mx, vx, z, ls, sf, psi1, psi2);
    GPX_CHECK_LAUNCH();
  }
  return GPX_OK;
}

// Adjoint of gpx_psi_fwd given dL/dpsi1 (N x M) and dL/dpsi2 (N x M x M), symmetric or (sym = 0)
// any: dsf2 (1, w.r.t. sf2), dell (Q, w.r.t. ell = exp(ls)), dZ (M x Q), dmx, dvx (N x Q).
long gpx_psi_bwd_gen_workspace(int N, int M, int Q) {
  return N < 1 ? 0 : (long)psi_bwd_blocks(N, M) * (M * Q + Q + 2);
}

int gpx_psi_bwd_gen(int N, int M, int Q, int sym, const double *mx, const double *vx, const double *z,
                    const double *ls, const double *sf, const double *dpsi1, const double *psi1,
                    const double *dpsi2, const double *psi2, double *dsf2, double *dell, double *dZ,
                    double *dmx, double *dvx, double *work, void *stream) {
  if (N < 1 || M < 1 || M > 256 || Q < 1 || Q > GPX_QMAX) return GPX_EINVAL;
  if (!mx || !vx || !z || !ls || !sf || !dpsi1 || !psi1 || !dpsi2 || !psi2 || !work) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const int blocks = psi_bwd_blocks(N, M);
  int rc;
#define PSI_GO(TN, W) \
  psi_bwd_launch<TN, W>(blocks, N, M, Q, sym, mx, vx, z, ls, dpsi1, psi1, dpsi2, psi2, dmx, dvx, work, st)
  if (M <= 64) rc = PSI_GO(1, 4);
  else if (M <= 128) rc = PSI_GO(2, 4);
  else rc = PSI_GO(2, 8);
#undef PSI_GO
  if (rc != GPX_OK) return rc;
  hipLaunchKernelGGL(psi_bwd_sum_kernel, dim3(gpx_cdiv(M * Q + Q + 1, 32)), dim3(256), 0, st, M, Q, blocks,
                     (const double *)work, sf, dsf2, dell, dZ);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// The same for a symmetric dpsi2; its workspace query covers N M^2 doubles as well, which callers
// of this entry point may count on having reserved.
long gpx_psi_bwd_workspace(int N, int M, int Q) { return (long)N * M * M + gpx_psi_bwd_gen_workspace(N, M, Q); }

int gpx_psi_bwd(int N, int M, int Q, const double *mx, const double *vx, const double *z,
                const double *ls, const double *sf, const double *dpsi1, const double *psi1,
                const double *dpsi2, const double *psi2, double *dsf2, double *dell, double *dZ,
                double *dmx, double *dvx, double *work, void *stream) {
  return gpx_psi_bwd_gen(N, M, Q, 1, mx, vx, z, ls, sf, dpsi1, psi1, dpsi2, psi2, dsf2, dell, dZ, dmx, dvx, work,
                         stream);
}

}  // extern "C"
