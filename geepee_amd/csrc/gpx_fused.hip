// Fused moment-matched (uncertain-input) layer: psi2 is never written to HBM.
//
// With d = 1/(2v+l), (mu - (z_a+z_b)/2)^2 = (mu-z_a)^2/2 + (mu-z_b)^2/2 - (z_a-z_b)^2/4 turns the
// psi2 exponent (kernels.py:219-223) into
//   log psi2[n,a,b] - 4 sf = u_na + u_nb - sum_q w_nq (z_aq - z_bq)^2,
//   u_na = sum_q [log(l d)/4 - d (mu-z_a)^2/2],  w_nq = (1/l - d)/4 = v d / (2 l),
// a sum of non-positive terms (no cancellation), so each 16 (pairs) x 16 (points) block of
// exponents is an FP64 MFMA product of K = Q cross terms on top of u_na + u_nb as the
// initial accumulator, followed by one exp per entry on the vector ALUs, and the result
// feeds the next MFMA contraction in the register layout the matrix core produced it in.
// (Expanding the square into K = 2Q + 2 features took 5 MFMAs at Q = 8 where this takes 2.)
//
// Pairs are visited as 16x16 tiles (A <= B) of the M x M square; a tile is processed in
// 16 "row blocks" (fixed a, 16 consecutive b).  Off-diagonal tiles count each unordered
// pair once with weight 2; diagonal tiles hold the full square with weight 1.
//
// Forward (aep_models.py:182-199): v[n,d] = sf2 + sum_ab Bhat[d,a,b] psi2[n,a,b] - m^2.
// Backward (aep_models.py:201-304 with kernels.py:302-444): per point the statistics
// T_na = sum_b L_nab and V_nq = sum_ab L_nab z_aq z_bq of L = dpsi2 * psi2, and over the
// points dBhat[d] = sum_n dv_nd psi2_n, Lsum = sum_n L_n, W_q = sum_n L_n d_nq, where
// dpsi2_n = sum_d dv_nd Bsym[d].
#include "gpx_frag.h"

#include <algorithm>

#include <mutex>

#define FQ_MAX 16
#define FM_MAX 256
#define U_PAD -1.0e4  // u of a padding point or column: its exp is an exact 0

// u no lower than U_PAD (a NaN stays): psi2 of a point so far out is an exact 0 either way, and
// the exponent of an infinite or huge mean or variance stays within what gpx_exp_tab reduces.
__device__ __forceinline__ double u_floor(double u) { return u < U_PAD ? U_PAD : u; }

// w = (1/l - d)/4 = v d / (2 l), with its limit at an infinite v (where v d is inf * 0).
__device__ __forceinline__ double cross_weight(double v, double d, double l) {
  return isinf(v) ? 0.25 / l : 0.5 * v * d / l;
}

namespace {

__device__ __forceinline__ void decode_tile(int t, int T, int &A, int &B) {
  A = 0;
  int rem = t;
  while (rem >= T - A) {
    rem -= T - A;
    ++A;
  }
  B = A + rem;
}

// Work items (point block, split) of the forward on a 1-D grid.
// Workgroups are dealt to the 8 XCDs round-robin by linear index; when the split count S
// divides 8, every block on XCD x serves split x mod S, so that XCD's L2 holds only that
// split's share of B-hat rather than all of it.  Returns false
// for the blocks past the last point block (a whole workgroup, before any barrier).
__device__ __forceinline__ bool split_block(int nblk, int S, int &pb, int &split) {
  const int id = blockIdx.x;
  if (8 % S == 0) {
    const int x = id & 7, per = 8 / S;
    split = x % S;
    pb = (id >> 3) * per + x / S;
  } else {
    split = id / nblk;
    pb = id - split * nblk;
  }
  return pb < nblk;
}
inline unsigned split_grid(long nblk, int S) {
  return (8 % S == 0) ? 8u * gpx_cdiv(nblk, 8 / S) : (unsigned)(nblk * S);
}

// Slots of the adjoint's per-point partials: one T slot per tile column, one V slot per tile.
inline int fused_t_slots(int M) { return (M + 15) / 16; }
inline int fused_v_slots(int M) {
  const int T = (M + 15) / 16;
  return T * (T + 1) / 2;
}

// ---------------------------------------------------------------------------
// forward: part[s][n][d] = sum over the tiles of split s of w * Bp[a,b,d] psi2[n,a,b]
// One block = NSUB x 16 points; the Bp loads of a row block are shared by the NSUB
// point tiles.  Bp is the symmetrised Bhat in pair-major layout (M x M x D) so the D
// values of a pair are contiguous.  z and u of the block's points lie in LDS
// (fwd_lds); off-diagonal tiles come first and their sums are doubled once.
//
// What bounds it: per row block and point tile KS + 4 DB MFMAs of 64 cycles plus about 225
// cycles of exps and adds on the same SIMD (55% of that rate reached at N = 4096, M = 128,
// Q = 8, D = 32: the rest is B-hat from the L2 and the set-up of u).  Forward entry,
// microseconds, expanded-square exponent -> this one: that shape 152 -> 106; 9999, 200, 4, 4
// 377 -> 285; 3001, 190, 10, 12 256 -> 133; 500, 200, 8, 16 77 -> 49; 300, 100, 5, 8 34 -> 27.
// ---------------------------------------------------------------------------
// Doubles of dynamic LDS: z (M x (4 KS + 1), columns past Q zero), u (16 T x 16 NSUB), and per
// point mu, d, w and log(l d)/4 (4 KS each); the final sum over the waves reuses it.
inline long fwd_lds(int M, int D, int KS, int NSUB) {
  const int T = (M + 15) / 16, pts = 16 * NSUB;
  const long n = (long)M * (4 * KS + 1) + 16L * T * pts + 4L * pts * 4 * KS, red = 4L * (D > 16 ? 32 : 16) * 17;
  return n > red ? n : red;
}

// Dynamic LDS up to which the requested points per workgroup are kept.
constexpr size_t kFwdLds = 100 << 10;

// KS: the 4-wide slices of the Q cross terms, ceil(Q / 4).
template <int DB, int NSUB, int KS>
__global__ __launch_bounds__(256) void fused_fwd_kernel(int N, int M, int Q, int D,
                                                        const double *__restrict__ mx,
                                                        const double *__restrict__ vx,
                                                        const double *__restrict__ z,
                                                        const double *__restrict__ ls,
                                                        const double *__restrict__ sf,
                                                        const double *__restrict__ Bp, int S,
                                                        double *__restrict__ part) {
  // DB = 0: D <= 4, the contraction with Bp as per-lane FMAs over the lane's four pair
  // columns (summed over the four lane rows once, at the end) instead of MFMAs that would
  // fill 4 of their 16 output rows
  constexpr bool VS = DB == 0;
  constexpr int DBA = VS ? 1 : DB, QP = 4 * KS, ZS = QP + 1, PTS = 16 * NSUB;
  extern __shared__ double dyn[];
  __shared__ double lam[FQ_MAX];
  __shared__ double etab[32];
  const int T = (M + 15) / 16, ntiles = T * (T + 1) / 2;
  double *zs = dyn, *us = zs + M * ZS, *pmu = us + 16 * T * PTS, *pd = pmu + PTS * QP, *pw = pd + PTS * QP,
         *pl = pw + PTS * QP;
  double (*red)[DBA * 16][17] = reinterpret_cast<double (*)[DBA * 16][17]>(dyn);
  int pb, split;
  if (!split_block((N + PTS - 1) / PTS, S, pb, split)) return;
  const int n0 = pb * PTS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < QP) lam[tid] = tid < Q ? exp(2.0 * ls[tid]) : 1.0;
  for (int e = tid; e < M * QP; e += 256) {
    const int m = e / QP, q = e % QP;
    zs[m * ZS + q] = q < Q ? z[m * Q + q] : 0.0;
  }
  gpx_exp_table_init(etab);
  __syncthreads();
  for (int e = tid; e < PTS * QP; e += 256) {
    const int pt = e / QP, q = e % QP, n = min(n0 + pt, N - 1);
    const double v = q < Q ? vx[(long)n * Q + q] : 0.0, l = lam[q], dd = 1.0 / (2.0 * v + l);
    pmu[e] = q < Q ? mx[(long)n * Q + q] : 0.0;
    pd[e] = dd;
    pw[e] = cross_weight(v, dd, l);
    pl[e] = 0.25 * log(l * dd);  // columns past Q: log 1
  }
  __syncthreads();
  {
    // u of this thread's point (256 threads are whole groups of points) at every 256/PTS-th m
    const int pt = tid % PTS;
    double mu[QP], hd[QP], c = 0.0;
#pragma unroll
    for (int q = 0; q < QP; ++q) {
      mu[q] = pmu[pt * QP + q];
      hd[q] = -0.5 * pd[pt * QP + q];
      c += pl[pt * QP + q];
    }
    for (int m = tid / PTS; m < 16 * T; m += 256 / PTS) {
      double u = U_PAD;
      if (m < M && n0 + pt < N) {
        u = c;
#pragma unroll
        for (int q = 0; q < QP; ++q) {
          const double dz = mu[q] - zs[m * ZS + q];  // columns past Q: both zero
          u = fma(hd[q] * dz, dz, u);
        }
        u = u_floor(u);
      }
      us[m * PTS + pt] = u;
    }
  }
  __syncthreads();
  const int ka = lane & 15, kq = lane >> 4;
  double bf[NSUB][KS];
#pragma unroll
  for (int u = 0; u < NSUB; ++u)
#pragma unroll
    for (int s = 0; s < KS; ++s) bf[u][s] = pw[(16 * u + ka) * QP + kq + 4 * s];
  gpx_d4 acc[NSUB][DBA];
#pragma unroll
  for (int u = 0; u < NSUB; ++u)
#pragma unroll
    for (int i = 0; i < DBA; ++i) acc[u][i] = gpx_d4{0.0, 0.0, 0.0, 0.0};
  // rows i = wave, wave + 4, ... of tile (A, B)
  auto tile = [&](int A, int B) {
    // column of this lane, clamped for the loads (a padding column's u is U_PAD)
    const int jl = min(16 * B + ka, M - 1);
    double zb[KS], ub[NSUB][4];
#pragma unroll
    for (int s = 0; s < KS; ++s) zb[s] = zs[jl * ZS + kq + 4 * s];
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) ub[u][r] = us[(16 * B + kq + 4 * r) * PTS + 16 * u + ka];
    for (int i = wave; i < 16; i += 4) {
      const int a = 16 * A + i;
      if (a >= M) break;
      // unconditional loads (column b and row d clamped; rows d >= D of acc are never
      // stored), issued together and waited for once
      // MFMA form: lane (d = 16 db + lane%16, b = lane/16 + 4r); VS: lane (b = lane/16 + 4r,
      // d < 4), the four rows of lane/16 reading the same values
      double bv[DBA][4], bs4[VS ? 4 : 1][4];
      if constexpr (VS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int b = min(16 * B + kq + 4 * r, M - 1);
#pragma unroll
          for (int d = 0; d < 4; ++d) bs4[r][d] = Bp[((long)a * M + b) * D + min(d, D - 1)];
        }
      } else {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int d = min(16 * db + ka, D - 1), b = min(16 * B + kq + 4 * r, M - 1);
            bv[db][r] = Bp[((long)a * M + b) * D + d];
          }
      }
      double af[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const double dz = zs[a * ZS + kq + 4 * s] - zb[s];
        af[s] = -dz * dz;
      }
#pragma unroll
      for (int u = 0; u < NSUB; ++u) {
        const double ua = us[a * PTS + 16 * u + ka];
        gpx_d4 e;
#pragma unroll
        for (int r = 0; r < 4; ++r) e[r] = ua + ub[u][r];
#pragma unroll
        for (int s = 0; s < KS; ++s) e = gpx_mfma16(af[s], bf[u][s], e);
        double p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = gpx_exp_tab(e[r], etab);
        if constexpr (VS) {
          // acc[u][0][d]: this lane's partial of part[n = lane%16][d] over its pair columns
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int d = 0; d < 4; ++d) acc[u][0][d] = fma(bs4[r][d], p[r], acc[u][0][d]);
        } else {
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[u][db] = gpx_mfma16(bv[db][r], p[r], acc[u][db]);
        }
      }
    }
  };
  // tiles split, split + S, ... of the off-diagonal ones in row order, then of the diagonal
  // ones, continuing the deal where the off-diagonal tiles ended
  const int noff = ntiles - T;
  for (int t = split; t < noff; t += S) {
    int A = 0, rem = t;
    while (rem >= T - 1 - A) rem -= T - 1 - A++;
    tile(A, A + 1 + rem);
  }
#pragma unroll
  for (int u = 0; u < NSUB; ++u)
#pragma unroll
    for (int i = 0; i < DBA; ++i) acc[u][i] *= 2.0;
  for (int t = (split + S - noff % S) % S; t < T; t += S) tile(t, t);
  const double sf2 = exp(2.0 * sf[0]), sf4 = sf2 * sf2;
  __syncthreads();  // red overlays z and u
#pragma unroll
  for (int u = 0; u < NSUB; ++u) {
    if constexpr (VS) {
      // the four lane rows summed (fixed order), then rows d < 4 of the block sum below
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const double t = gpx_swap_add<16>(gpx_swap_add<32>(acc[u][0][d]));
        if (kq == 0) red[wave][d][ka] = t;
      }
    } else {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][db * 16 + kq + 4 * r][ka] = acc[u][db][r];
    }
    __syncthreads();
    for (int idx = tid; idx < (VS ? 4 : DB * 16) * 16; idx += 256) {
      const int dd = idx >> 4, nn = idx & 15, n = n0 + 16 * u + nn;
      const double s = red[0][dd][nn] + red[1][dd][nn] + red[2][dd][nn] + red[3][dd][nn];
      if (dd < D && n < N) part[((long)split * N + n) * D + dd] = sf4 * s;
    }
    __syncthreads();
  }
}

// out[(a*M + b)*D + d] = (B[d,a,b] + B[d,b,a]) / 2
__global__ void sym_pairmajor_kernel(int D, int M, const double *__restrict__ B, double *__restrict__ out) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const long MM = (long)M * M;
  if (e >= D * MM) return;
  const long ab = e / D;
  const int d = (int)(e % D), a = (int)(ab / M), b = (int)(ab % M);
  out[e] = 0.5 * (B[d * MM + (long)a * M + b] + B[d * MM + (long)b * M + a]);
}


// Point features of the adjoint, formed once per launch: pf[n] = [w_n (16, zero past Q) | 1 |
// d_n (15, zero past Q)] and u[n][m].  PF_PTS points per workgroup: its set-up (a log and a
// division per dimension) and M Q multiply-adds per point are latency, hidden by many workgroups
// (16 points in each: N = 3001, M = 190, Q = 10 12.6 -> 7.3 us).
constexpr int PF_W = 32, PF_PTS = 4;

__global__ __launch_bounds__(256) void fused_point_feat_kernel(int N, int M, int Q, const double *__restrict__ mx,
                                                               const double *__restrict__ vx,
                                                               const double *__restrict__ z,
                                                               const double *__restrict__ ls,
                                                               double *__restrict__ pf, double *__restrict__ un) {
  __shared__ double mu[PF_PTS][FQ_MAX], dd[PF_PTS][FQ_MAX], lg[PF_PTS][FQ_MAX];
  const int tid = threadIdx.x, n0 = blockIdx.x * PF_PTS;
  if (tid < PF_PTS * 16) {
    const int nn = tid >> 4, q = tid & 15, n = n0 + nn;
    const bool in = q < Q && n < N;
    const double lam = q < Q ? exp(2.0 * ls[q]) : 1.0;
    const double v = in ? vx[(long)n * Q + q] : 0.0, d = 1.0 / (2.0 * v + lam);
    mu[nn][q] = in ? mx[(long)n * Q + q] : 0.0;
    dd[nn][q] = -0.5 * d;
    lg[nn][q] = in ? 0.25 * log(lam * d) : 0.0;
    if (n < N) {
      double *o = pf + (long)n * PF_W;
      o[q] = in ? cross_weight(v, d, lam) : 0.0;
      if (q < 15) o[17 + q] = in ? d : 0.0;
      else o[16] = 1.0;
    }
  }
  __syncthreads();
  for (int e = tid; e < PF_PTS * M; e += 256) {
    const int i = e / M, m = e % M;
    if (n0 + i >= N) break;
    double u = 0.0;
    for (int k = 0; k < Q; ++k) u += lg[i][k];
#pragma unroll 4
    for (int k = 0; k < Q; ++k) {
      const double dz = mu[i][k] - z[m * Q + k];
      u = fma(dd[i][k] * dz, dz, u);
    }
    un[(long)(n0 + i) * M + m] = u_floor(u);
  }
}

// Row k of a staged 16 x 32 dv block keeps column c at c ^ dv_swizzle(k).  The two read
// patterns (16 rows x 4 columns, and 4 rows x 16 columns) then fall on distinct LDS banks
// two lanes a bank: rows k and k+8 share their column permutation, and of every four
// consecutive rows two keep the halves of the row in place and two swap them.
__device__ __forceinline__ int dv_swizzle(int k) { return 4 * (((k & 1) << 2) | ((k >> 1) & 3)); }

// Wave-scope ordering of LDS accesses (a wave reading what its other lanes wrote).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// backward: the per-pair sums over the points of a range
//   dBhat[d, a, b] = sum_n dv_nd psi2_nab,  LW[a, b, q'] = sum_n [1 | d_nq'] L_nab
// and the per-point sums over the pairs from one evaluation of p and G per (point, pair).
// A workgroup of MG_NW = 8 waves owns the 16 rows of one tile (A, B) over one point range;
// wave w holds rows a = 16A + w + 8u (u < 2).  Per row and 16-point block: the exponent,
// G = <dv, B-hat>, p, L = G p and the dB-hat / LW contractions, and
//   U[n][q'] = sum_b L[n][b] [1 | z_b][q']  (L transposed through the wave's LDS, 4 MFMAs)
//   row sums  T[n][a] = U[n][0]                      -> Tpart slot B, column a
//   V[n][q]  += w z_aq U[n][1+q]  (w = 2 off the diagonal tile, 1 on it)
// and per workgroup (A < B) the column sums sum_a L[n][a][b] -> Tpart slot A, column b.
// Column c of tile C thus has exactly T slots (row sums from tiles (C, s), s >= C; column
// sums from tiles (s, C), s < C), each written once; V has one slot per tile.  The
// 8-wave sums of the column sums and V go through LDS in wave order (double-buffered
// by block parity, so one barrier per block serves the staging and both sums); a block's
// sums are read and written out during the next block, beside its first MFMAs.
// DS = ceil(D / 4) for D <= 16, 8 up to 32; KS = ceil(Q / 4); G = ceil((Q + 1) / 4).
// ---------------------------------------------------------------------------
//
// What bounds it: per row and block 64 (KS + 2 DS + 2 G) cycles of MFMAs (the dB-hat, LW and U products
// as 4 x 4 x 4 forms of only the rows and columns there are, where 16 x 16 tiles were up to three
// quarters padding; not at D > 16, whose registers hold no operands for them) and about 230 of
// exps and other FP64 vector work on the same SIMD, which add up, and the LDS reads of operands;
// two waves per SIMD (LDS and registers hold one workgroup per CU; four at 128 registers spilled
// and took 1882 us in place of 711).  Adjoint entry, microseconds, expanded-square exponent ->
// now: N = 4096, M = 128, Q = 8, D = 32 300 -> 255; 9999, 200, 4, 4 927 -> 610; 3001, 190, 10, 12
// 421 -> 305; 500, 200, 8, 16 200 -> 118.
constexpr int MG_NW = 8;

// D += A B of the 16 x 16 x 4 MFMA on four doubles in place.
__device__ __forceinline__ void mfma16_at(double a, double b, double *d) {
  const gpx_d4 t = gpx_mfma16(a, b, gpx_d4{d[0], d[1], d[2], d[3]});
#pragma unroll
  for (int r = 0; r < 4; ++r) d[r] = t[r];
}

template <int DS, int KS, int G>
__global__ __launch_bounds__(64 * MG_NW) void fused_bwd_merged_kernel(
    int N, int M, int Q, int D, const double *__restrict__ z, const double *__restrict__ sf,
    const double *__restrict__ Bp, const double *__restrict__ dv, const double *__restrict__ pf,
    const double *__restrict__ un, int nsplit, int nchunk, double *__restrict__ dBpart,
    double *__restrict__ LWpart, double *__restrict__ Tpart, double *__restrict__ Vpart) {
  constexpr int NR = 2;
  // 4 x 4 MFMA forms where they need fewer than a 16-row tile's rows: of U and LW (G groups of
  // four columns q'), of dB-hat (DS groups of four rows d)
  constexpr bool U4 = G < 4 && DS < 8, D4 = DS < 4;
  constexpr int DB = DS > 4 ? 2 : 1, UC = U4 ? G : 4, LR = U4 ? G : 4, DR = D4 ? DS : 4 * DB;
  __shared__ double pfs[2][16][PF_W + 2];      // point features
  __shared__ double lus[2][16][PF_W + 1];      // u at the tile's rows (16) and columns (16)
  __shared__ double dvs[2][16][32];
  __shared__ double trn[MG_NW][NR][16][17];    // per-wave transposes of L
  __shared__ double csum[2][MG_NW][16][17];    // per-wave column sums  [n][b]
  __shared__ double vsum[2][MG_NW][16][(DS < 8 ? 4 * G : 16) + 1];  // per-wave V terms   [n][q']
  // the exponent's pair operands of the wave's rows, in LDS where D > 16 leaves no registers
  constexpr bool AF_LDS = DB == 2;
  __shared__ double afs[AF_LDS ? MG_NW : 1][NR][KS][AF_LDS ? 64 : 1];
  __shared__ double etab[32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T = (M + 15) / 16;
  const int tile = blockIdx.x;
  int A, B;
  decode_tile(tile, T, A, B);
  const bool off = A != B;
  const int ns = blockIdx.y;
  const int nbeg = ns * nchunk, nend = min(N, nbeg + nchunk);
  const int ka = lane & 15, kq = lane >> 4;
  const int jb = 16 * B + ka;
  const double sf2 = exp(2.0 * sf[0]), sf4 = sf2 * sf2;
  int a[NR];
  bool act[NR];
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    a[u] = 16 * A + wave + 8 * u;
    act[u] = a[u] < M;
  }
  // pair operands of the wave's rows: -(z_a - z_b)^2 (k = kq + 4s), sf4 B-hat, the V weight
  double af[AF_LDS ? 1 : NR][KS], bs[NR][DS], zw[NR][U4 ? G : 1];
  const int k4 = lane & 3, n4 = 4 * ((lane >> 2) & 3) + kq;  // 4 x 4 results: column k4, row n4
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    const bool bv = jb < M && act[u];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = kq + 4 * s;
      const double dz = bv && k < Q ? z[a[u] * Q + k] - z[jb * Q + k] : 0.0;
      if constexpr (AF_LDS) afs[wave][u][s][lane] = -dz * dz; else af[u][s] = -dz * dz;
    }
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const int d = kq + 4 * s;
      bs[u][s] = (bv && d < D) ? sf4 * Bp[((long)a[u] * M + jb) * D + d] : 0.0;
    }
    // V weight of this lane's columns q' of U: w z_a[q'-1]
#pragma unroll
    for (int g = 0; g < (U4 ? G : 1); ++g) {
      const int q = U4 ? 4 * g + k4 : ka;
      zw[u][g] = (act[u] && q >= 1 && q <= Q) ? (off ? 2.0 : 1.0) * z[a[u] * Q + q - 1] : 0.0;
    }
  }
  // B operand of U: [1 | z_b] for b = 16B + kq + 4s (rows), q' (columns); padding
  // columns b >= M give zeros (their L is 0 as well)
  double zx[4][U4 ? G : 1];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int g = 0; g < (U4 ? G : 1); ++g) {
      const int b = 16 * B + kq + 4 * s, q = U4 ? 4 * g + k4 : ka;
      zx[s][g] = (b < M && q <= Q) ? (q == 0 ? 1.0 : z[b * Q + q - 1]) : 0.0;
    }
  // rows d = 4 i + kq of dacc[i], q' = 4 i + kq of lacc[i], column b = ka
  double dacc[NR][DR], lacc[NR][LR];
#pragma unroll
  for (int u = 0; u < NR; ++u) {
#pragma unroll
    for (int i = 0; i < LR; ++i) lacc[u][i] = 0.0;
#pragma unroll
    for (int i = 0; i < DR; ++i) dacc[u][i] = 0.0;
  }
  // staging: thread (row sk < 16, column sc < 32) of each of the three arrays
  const int sk = tid >> 5, sc = tid & 31;
  const int lcol = sc < 16 ? 16 * A + sc : 16 * B + sc - 16;
  double rp, rl, rd;
  auto fetch = [&](int n0) {
    const bool in = n0 + sk < nend;
    rp = in ? pf[(long)(n0 + sk) * PF_W + sc] : 0.0;
    rl = in && lcol < M ? un[(long)(n0 + sk) * M + lcol] : U_PAD;
    rd = in && sc < D ? dv[(long)(n0 + sk) * D + sc] : 0.0;
  };
  auto stage = [&](int buf) {
    pfs[buf][sk][sc] = rp;
    lus[buf][sk][sc] = rl;
    dvs[buf][sk][sc ^ dv_swizzle(sk)] = rd;
  };
  // the 8-wave sums of block n0's column sums and V terms (buffer cb), written out
  auto reduce = [&](int n0, int cb) {
    if (tid < 256) {
      const int nn = tid >> 4, bb = tid & 15, n = n0 + nn, b = 16 * B + bb;
      if (off && n < nend && b < M) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < MG_NW; ++w) t += csum[cb][w][nn][bb];
        Tpart[((long)A * N + n) * M + b] = t;
      }
    } else {
      const int e = tid - 256, nn = e >> 4, qq = e & 15, n = n0 + nn;
      if (qq >= 1 && qq <= Q && n < nend) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < MG_NW; ++w) v += vsum[cb][w][nn][qq];
        Vpart[((long)tile * N + n) * Q + qq - 1] = v;
      }
    }
  };
  fetch(nbeg);
  stage(0);
  gpx_exp_table_init(etab);
  __syncthreads();
  const int swa = dv_swizzle(ka);
  int buf = 0;
  for (int n0 = nbeg; n0 < nend; n0 += 16) {
    const bool more = n0 + 16 < nend;  // uniform over the workgroup
    if (more) fetch(n0 + 16);
    double pa[KS], da[DS], dvv[4][D4 ? DS : DB], dq[4][U4 ? G : 1], ub[4];
#pragma unroll
    for (int s = 0; s < KS; ++s) pa[s] = pfs[buf][ka][kq + 4 * s];
#pragma unroll
    for (int r = 0; r < 4; ++r) ub[r] = lus[buf][kq + 4 * r][16 + ka];
#pragma unroll
    for (int s = 0; s < DS; ++s) da[s] = dvs[buf][ka][(kq + 4 * s) ^ swa];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = kq + 4 * r;
#pragma unroll
      for (int i = 0; i < (D4 ? DS : DB); ++i)
        dvv[r][i] = dvs[buf][k][(D4 ? 4 * i + k4 : 16 * i + ka) ^ dv_swizzle(k)];
#pragma unroll
      for (int i = 0; i < (U4 ? G : 1); ++i) dq[r][i] = pfs[buf][k][16 + (U4 ? 4 * i + k4 : ka)];
    }
    double cs[4] = {0.0, 0.0, 0.0, 0.0}, vw[UC];
#pragma unroll
    for (int i = 0; i < UC; ++i) vw[i] = 0.0;
    // both rows in step, without a branch (rows past M carry zeros), so that one's latencies
    // hide behind the other's work
    gpx_d4 e[NR], g[NR];
#pragma unroll
    for (int u = 0; u < NR; ++u) {
#pragma unroll
      for (int r = 0; r < 4; ++r) e[u][r] = ub[r] + lus[buf][kq + 4 * r][wave + 8 * u];
      g[u] = gpx_d4{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        double f;
        if constexpr (AF_LDS) f = afs[wave][u][s][lane]; else f = af[u][s];
        e[u] = gpx_mfma16(pa[s], f, e[u]);
      }
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int u = 0; u < NR; ++u) g[u] = gpx_mfma16(da[s], bs[u][s], g[u]);
    // the previous block's 8-wave sums, while this block's first MFMAs run (its buffer
    // half is not written again before the next barrier)
    if (n0 > nbeg) reduce(n0 - 16, buf ^ 1);
    double p[NR][4], L[NR][4];
#pragma unroll
    for (int u = 0; u < NR; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[u][r] = gpx_exp_tab(e[u][r], etab);
        L[u][r] = g[u][r] * p[u][r];
        cs[r] += L[u][r];
        // L (lane: n = kq + 4r, b = ka) to the A-operand layout (lane: n = ka, b = kq + 4s)
        // through the wave's LDS
        trn[wave][u][kq + 4 * r][ka] = L[u][r];
      }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        if constexpr (D4) {
#pragma unroll
          for (int i = 0; i < DS; ++i) dacc[u][i] = gpx_mfma4(dvv[r][i], p[u][r], dacc[u][i]);
        } else {
#pragma unroll
          for (int i = 0; i < DB; ++i) mfma16_at(dvv[r][i], p[u][r], dacc[u] + 4 * i);
        }
        if constexpr (U4) {
#pragma unroll
          for (int i = 0; i < G; ++i) lacc[u][i] = gpx_mfma4(dq[r][i], L[u][r], lacc[u][i]);
        } else {
          mfma16_at(dq[r][0], L[u][r], lacc[u]);
        }
      }
    // U = L [1 | z_b]
    double lt[NR][4];
#pragma unroll
    for (int u = 0; u < NR; ++u)
#pragma unroll
      for (int s = 0; s < 4; ++s) lt[u][s] = trn[wave][u][ka][kq + 4 * s];
    if constexpr (U4) {  // lane holds U[n = n4][q' = 4 i + k4]
      double U[NR][G];
#pragma unroll
      for (int u = 0; u < NR; ++u)
#pragma unroll
        for (int i = 0; i < G; ++i) U[u][i] = 0.0;
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int u = 0; u < NR; ++u)
#pragma unroll
          for (int i = 0; i < G; ++i) U[u][i] = gpx_mfma4(lt[u][s], zx[s][i], U[u][i]);
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        if (k4 == 0 && act[u] && n0 + n4 < nend) Tpart[((long)B * N + n0 + n4) * M + a[u]] = U[u][0];
#pragma unroll
        for (int i = 0; i < G; ++i) vw[i] += zw[u][i] * U[u][i];
      }
    } else {  // U[n = kq + 4r][q' = ka]
      gpx_d4 U[NR];
#pragma unroll
      for (int u = 0; u < NR; ++u) U[u] = gpx_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int u = 0; u < NR; ++u) U[u] = gpx_mfma16(lt[u][s], zx[s][0], U[u]);
#pragma unroll
      for (int u = 0; u < NR; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + kq + 4 * r;
          if (ka == 0 && act[u] && n < nend) Tpart[((long)B * N + n) * M + a[u]] = U[u][r];
          vw[r] += zw[u][0] * U[u][r];
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) csum[buf][wave][kq + 4 * r][ka] = cs[r];
#pragma unroll
    for (int i = 0; i < UC; ++i) {
      if constexpr (U4) vsum[buf][wave][n4][4 * i + k4] = vw[i]; else vsum[buf][wave][kq + 4 * i][ka] = vw[i];
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  if (nend > nbeg) reduce(nbeg + (nend - nbeg - 1) / 16 * 16, buf ^ 1);  // the last block's
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    if (!act[u]) continue;
#pragma unroll
    for (int i = 0; i < DR; ++i) {
      const int d = 4 * i + kq;
      if (d < D && jb < M) dBpart[(((long)ns * D + d) * M + a[u]) * M + jb] = sf4 * dacc[u][i];
    }
#pragma unroll
    for (int i = 0; i < LR; ++i) {
      const int qq = 4 * i + kq;
      if (qq <= Q && jb < M) LWpart[(((long)ns * M + a[u]) * M + jb) * (Q + 1) + qq] = lacc[u][i];
    }
  }
}

// Sum of the adjoint kernel's point-range partials.  One workgroup per stored 16 x 16
// tile pair (A <= B, the half the pair kernel writes) and output slice (k < D: dBhat[k],
// k >= D: column q = k - D of LW), 256 entries each; rows are read coalesced and the
// mirrored tile (B, A) is written through an LDS transpose.  dBhat (D x M x M) and LW
// ((M*M) x (Q+1)) come out in the layouts of the materialising path.
__global__ __launch_bounds__(256) void fused_pairs_finish(int M, int Q, int D, int nsplit,
                                                          const double *__restrict__ dBpart,
                                                          const double *__restrict__ LWpart,
                                                          double *__restrict__ dBhat, double *__restrict__ LW) {
  __shared__ double tile[16][17];
  const int T = (M + 15) / 16;
  int t = blockIdx.x, A = 0;
  while (t >= T - A) {
    t -= T - A;
    ++A;
  }
  const int B = A + t, k = blockIdx.y, tid = threadIdx.x, i = tid >> 4, j = tid & 15;
  const long MM = (long)M * M;
  const int a = A * 16 + i, b = B * 16 + j;
  if (k < D) {
    double s = 0.0;
    if (a < M && b < M) {
#pragma unroll 8
      for (int p = 0; p < nsplit; ++p) s += dBpart[(((long)p * D + k) * M + a) * M + b];
      dBhat[k * MM + (long)a * M + b] = s;
    }
    if (A != B) {
      tile[i][j] = s;
      __syncthreads();
      const int a2 = B * 16 + i, b2 = A * 16 + j;
      if (a2 < M && b2 < M) dBhat[k * MM + (long)a2 * M + b2] = tile[j][i];
    }
  } else {
    const int Q1 = Q + 1, q = k - D;
    if (a < M && b < M) {
      double s = 0.0;
#pragma unroll 8
      for (int p = 0; p < nsplit; ++p) s += LWpart[(((long)p * M + a) * M + b) * Q1 + q];
      LW[((long)a * M + b) * Q1 + q] = s;
      if (A != B) LW[((long)b * M + a) * Q1 + q] = s;
    }
  }
}


// Per-point finish of the fused adjoint, a workgroup per point, point after point: T = the sum of
// the S slots of Tpart, V of the SV slots of Vpart, Lp = dpsi1 psi1, then dmx, dvx and the point's
// share of dell, and, in registers over the workgroup's points, what T and Lp give to dZ:
//   dZ_aq += T (2 d mu - z (d + 1/l)) - Lp e (z - mu),  d = 1/(2v+l), e = 1/(v+l)
// (the rest of dZ comes from the pair sums LW).  Lane (g, c) of wave w owns q = g + 4 r (r < KR) and
// the columns a = 16 (w + 4 j) + c; the lane groups share the slots, sums over a run across the 16
// lanes of a row, then over the waves through LDS.  Bound by reading the slots (13 N M doubles at
// M = 200).  With the tail below, in place of a wave per point that stored T and Lp for two
// products, two column sums and an assembly: whole adjoint, us, N = 3001, M = 190, Q = 10, D = 12
// 321 -> 299, 4096, 128, 8, 32 271 -> 266, 300, 100, 5, 8 58 -> 49, 150, 20, 4, 8 40 -> 30.
// part[block]: [dZ (M x Q) | sum of H (Q) | S0, A1].
constexpr int RF_RED = 5 * FQ_MAX + 2;

template <int KR, int MJ>  // MJ: column tiles of a wave, ceil(M / 64)
__global__ __launch_bounds__(256, 3) void fused_rows_finish(
    int N, int M, int Q, int S, int SV, const double *__restrict__ mx, const double *__restrict__ vx,
    const double *__restrict__ z, const double *__restrict__ ls, const double *__restrict__ Tpart,
    const double *__restrict__ Vpart, const double *__restrict__ dpsi1, const double *__restrict__ psi1,
    double *__restrict__ dmx, double *__restrict__ dvx, double *__restrict__ part) {
  constexpr int ZLD = 4 * KR + 1;
  extern __shared__ double rf_lds[];  // z, rows of ZLD
  __shared__ double red[2][4][RF_RED];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15, MT = (M + 15) >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int e = tid; e < M * ZLD; e += 256) rf_lds[e] = e % ZLD < Q ? z[e / ZLD * Q + e % ZLD] : 0.0;
  __syncthreads();
  double l[KR], il[KR], dz[MJ][KR], hsum = 0.0, s0sum = 0.0, a1sum = 0.0;
  int col[MJ];
  bool on[MJ];
#pragma unroll
  for (int r = 0; r < KR; ++r) {
    l[r] = g + 4 * r < Q ? exp(2.0 * ls[g + 4 * r]) : 1.0;
    il[r] = 1.0 / l[r];
  }
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int a = 16 * (w + 4 * j) + c;
    on[j] = a < M;
    col[j] = min(a, M - 1);
#pragma unroll
    for (int r = 0; r < KR; ++r) dz[j][r] = 0.0;
  }
  const int tn = (MT - w + 3) >> 2;  // this wave's column tiles (may be 0)
  const int tq = min(tid, Q - 1);
  const double ell = exp(ls[tq]), lq = exp(2.0 * ls[tq]);
  int par = 0;
  for (int n = blockIdx.x; n < N; n += gridDim.x, par ^= 1) {
    // every load at a clamped (valid) index, issued together; S <= 16, SV <= 136
    double tv[4][MJ], vv[3][KR], T[MJ], Lp[MJ], V[KR];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double *row = Tpart + ((long)min(g + 4 * i, S - 1) * N + n) * M;
#pragma unroll
      for (int j = 0; j < MJ; ++j) tv[i][j] = 4 * i < S && j < tn ? row[col[j]] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double *row = Vpart + ((long)min(16 * w + c + 64 * i, SV - 1) * N + n) * Q;
#pragma unroll
      for (int r = 0; r < KR; ++r) vv[i][r] = 64 * i < SV ? row[min(g + 4 * r, Q - 1)] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      const double x = dpsi1[(long)n * M + col[j]] * psi1[(long)n * M + col[j]];
      Lp[j] = on[j] ? x : 0.0;
      T[j] = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (g + 4 * i < S) T[j] += tv[i][j];
    }
#pragma unroll
    for (int r = 0; r < KR; ++r) {
      V[r] = 0.0;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (16 * w + c + 64 * i < SV) V[r] += vv[i][r];
    }
    double S0 = 0.0, A1 = 0.0;
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      if (j < tn) T[j] = gpx_swap_add<16>(gpx_swap_add<32>(T[j]));
      T[j] = on[j] ? T[j] : 0.0;
      S0 += T[j];
      A1 += Lp[j];
    }
    S0 = gpx_row_sum(S0);
    A1 = gpx_row_sum(A1);
    double *rw = red[par][w];
#pragma unroll
    for (int r = 0; r < KR; ++r) {
      const int q = g + 4 * r, qc = min(q, Q - 1);
      const double mu = mx[(long)n * Q + qc], v = vx[(long)n * Q + qc];
      const double d = gpx_recip(2.0 * v + l[r]), e = gpx_recip(v + l[r]);
      double S1 = 0.0, Z2 = 0.0, B1 = 0.0, C1 = 0.0;
#pragma unroll
      for (int j = 0; j < MJ; ++j) {
        if (j >= tn) break;
        const double zz = rf_lds[col[j] * ZLD + q], zm = zz - mu, tz = T[j] * zz, lz = Lp[j] * zm;
        S1 += tz;
        Z2 = fma(tz, zz, Z2);
        B1 += lz;
        C1 = fma(lz, zm, C1);
        dz[j][r] += d * (2.0 * mu * T[j] - tz) - il[r] * tz - e * lz;
      }
      S1 = gpx_row_sum(S1);
      Z2 = gpx_row_sum(Z2);
      B1 = gpx_row_sum(B1);
      C1 = gpx_row_sum(C1);
      const double Vq = gpx_row_sum(V[r]);
      if (c == 0) {
        rw[2 + q] = S1;
        rw[2 + FQ_MAX + q] = Z2;
        rw[2 + 2 * FQ_MAX + q] = Vq;
        rw[2 + 3 * FQ_MAX + q] = B1;
        rw[2 + 4 * FQ_MAX + q] = C1;
      }
    }
    if (lane == 0) {
      rw[0] = S0;
      rw[1] = A1;
    }
    __syncthreads();  // red[par] is next written two points on, behind the next point's barrier
    if (tid < Q) {
      const int q = tid;
      auto sum = [&](int i) { return red[par][0][i] + red[par][1][i] + red[par][2][i] + red[par][3][i]; };
      const double s0 = sum(0), a1 = sum(1), s1 = sum(2 + q), tz2 = sum(2 + FQ_MAX + q), vs = sum(2 + 2 * FQ_MAX + q),
                   b1 = sum(2 + 3 * FQ_MAX + q), c1 = sum(2 + 4 * FQ_MAX + q);
      const double m = mx[(long)n * Q + q], v = vx[(long)n * Q + q];
      const double d = 1.0 / (2.0 * v + lq), e = 1.0 / (v + lq);
      const double quad = m * m * s0 - 2.0 * m * s1 + 0.5 * (tz2 + vs);
      dmx[(long)n * Q + q] = -2.0 * d * (m * s0 - s1) + e * b1;
      dvx[(long)n * Q + q] = 2.0 * d * d * quad - d * s0 + 0.5 * e * (e * c1 - a1);
      hsum += 2.0 * ell * (v / lq * d * s0 + d * d * quad + (tz2 - vs) / (2.0 * lq * lq));
      hsum += e * ell * (e * c1 + v / lq * a1);
      s0sum += s0;
      a1sum += a1;
    }
  }
  double *po = part + (long)blockIdx.x * (M * Q + Q + 2);
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int r = 0; r < KR; ++r)
      if (on[j] && g + 4 * r < Q) po[col[j] * Q + g + 4 * r] = dz[j][r];
  if (tid < Q) po[M * Q + tid] = hsum;
  if (tid == 0) {
    po[M * Q + Q] = s0sum;
    po[M * Q + Q + 1] = a1sum;
  }
}

// The tail: dZ_a = the blocks' partials + sum_b (Lsum_ab / l - W_ab) z_b (one workgroup per a; LW
// ((M*M) x (Q+1)) = [Lsum | W]), and a last workgroup for dell and dsf2 = (A1 + 2 S0) / sf2.
__global__ __launch_bounds__(256) void fused_tail_kernel(int M, int Q, int blocks, const double *__restrict__ z,
                                                         const double *__restrict__ ls,
                                                         const double *__restrict__ sf,
                                                         const double *__restrict__ LW,
                                                         const double *__restrict__ part, double *__restrict__ dsf2,
                                                         double *__restrict__ dell, double *__restrict__ dZ) {
  __shared__ double red[16][17];
  const int a = blockIdx.x, tid = threadIdx.x, q = tid & 15, h = tid >> 4, width = M * Q + Q + 2;
  double s = 0.0;
  if (a < M && q < Q) {
    const double il = 1.0 / exp(2.0 * ls[q]);
    for (int b = h; b < M; b += 16) {
      const double *row = LW + ((long)a * M + b) * (Q + 1);
      s += (il * row[0] - row[1 + q]) * z[b * Q + q];
    }
  }
  // columns of the partials: dZ's row a, or [H | S0 | A1]
  const int cols = a < M ? Q : Q + 2;
  // (four running sums a thread: over up to 1024 blocks a single one let dell's error grow)
  double t4[4] = {0.0, 0.0, 0.0, 0.0}, x = 0.0;
  if (q < cols) {
#pragma unroll 4
    for (int k = h; k < blocks; k += 64)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double p = part[(long)min(k + 16 * u, blocks - 1) * width + a * Q + q];
        t4[u] += k + 16 * u < blocks ? p : 0.0;
      }
  }
  const double t = (t4[0] + t4[1]) + (t4[2] + t4[3]);
  if (a == M && q == 0 && Q + 1 == 16) {  // the 17th column, A1 at Q = 15
    for (int k = h; k < blocks; k += 16) x += part[(long)k * width + M * Q + 16];
  }
  red[h][q] = s + t;
  if (q == 0) red[h][16] = x;
  __syncthreads();
  if (tid > 16) return;
  double v = red[0][tid];
#pragma unroll
  for (int k = 1; k < 16; ++k) v += red[k][tid];
  if (a < M) {
    if (tid < Q) dZ[a * Q + tid] = v;
    return;
  }
  if (tid < Q) dell[tid] = v;
  red[0][tid] = v;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (tid == 0) dsf2[0] = (red[0][Q + 1] + 2.0 * red[0][Q]) / exp(2.0 * sf[0]);
}

// Workgroups of the row finish: as many as the registers let a CU hold (four where KR and MJ are
// small, else three), each with as many points as the others.
int rows_finish_blocks(int N, int M, int Q) {
  const int per = Q <= 4 || M <= 64 || (Q <= 8 && M <= 128) ? 1024 : 768;
  return (int)gpx_cdiv(N, gpx_cdiv(N, per));
}

// psi1, m = psi1 Ahat^T and v = sf2 + sum_s part - m^2 for FIN_PTS points per block (8: two waves
// per SIMD at N = 4096).  The means are products on the matrix cores, each wave every fourth group
// of 8 inducing points, added in wave order (a thread per output walked M inducing points with a
// row of Ahat of its own: N = 4096, M = 128, Q = 8, D = 32 21 -> 10 us, 3001, 190, 10, 12 16 -> 11).
// The split partials' loads issue four at a time (summed in split order).
constexpr int FIN_PTS = 8;

__global__ __launch_bounds__(256) void fused_fwd_finish(int N, int M, int Q, int D, const double *__restrict__ mx,
                                                        const double *__restrict__ vx,
                                                        const double *__restrict__ z,
                                                        const double *__restrict__ ls,
                                                        const double *__restrict__ sf,
                                                        const double *__restrict__ Ahat,
                                                        const double *__restrict__ part, int S,
                                                        double *__restrict__ psi1, double *__restrict__ mout,
                                                        double *__restrict__ vout) {
  __shared__ double p1[FIN_PTS][FM_MAX + 1];
  __shared__ double ms[4][2][FIN_PTS * 16];  // the waves' means
  __shared__ double rden[FIN_PTS][FQ_MAX], mus[FIN_PTS][FQ_MAX], lts[FIN_PTS][FQ_MAX], lcs[FIN_PTS];
  const int n0 = blockIdx.x * FIN_PTS, tid = threadIdx.x;
  const double sf2 = exp(2.0 * sf[0]);
  // per point and dimension (one thread each): 1 / (2 (v + l)), mx, and log(l / (l + v)) / 2,
  // whose sum over q (in q order) is the point's constant (independent of the inducing point)
  if (tid < FIN_PTS * Q) {
    const int nn = tid / Q, q = tid % Q, n = n0 + nn;
    const double l = exp(2.0 * ls[q]), v = n < N ? vx[(long)n * Q + q] : 0.0;
    rden[nn][q] = 1.0 / (2.0 * (v + l));
    mus[nn][q] = n < N ? mx[(long)n * Q + q] : 0.0;
    lts[nn][q] = 0.5 * log(l / (l + v));
  }
  __syncthreads();
  if (tid < FIN_PTS) {
    double lc = 0.0;
    for (int q = 0; q < Q; ++q) lc += lts[tid][q];
    lcs[tid] = lc;
  }
  __syncthreads();
  for (int e = tid; e < FIN_PTS * M; e += 256) {
    const int nn = e / M, m = e % M, n = n0 + nn;
    double val = 0.0;
    if (n < N) {
      double acc = 0.0;
      for (int q = 0; q < Q; ++q) {
        const double dlt = mus[nn][q] - z[m * Q + q];
        acc -= dlt * dlt * rden[nn][q];
      }
      val = sf2 * exp(acc + lcs[nn]);
      psi1[(long)n * M + m] = val;
    }
    p1[nn][m] = val;
  }
  __syncthreads();
  // m: rows are the points (past the last: the last again), columns the outputs
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
  const double *prow = p1[min(c, FIN_PTS - 1)];
  const int groups = M >> 3, kr = M & 7;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if (16 * t >= D) break;
    const GpxOperand<1, true> ob(Ahat, M, 16 * t, D, lane);
    gpx_d4 acc = {0.0, 0.0, 0.0, 0.0};
    GpxFrag<1> f;
    for (int k = w; k < groups; k += 4) {
      ob.load(f, 8 * k);
#pragma unroll
      for (int s = 0; s < 2; ++s) acc = gpx_mfma16(prow[8 * k + 2 * g + s], f.v[s][0], acc);
    }
    if (kr && w == groups % 4) {
      ob.load_tail(f, 8 * groups, kr, lane);
#pragma unroll
      for (int s = 0; s < 2; ++s)
        acc = gpx_mfma16(2 * g + s < kr ? prow[8 * groups + 2 * g + s] : 0.0, f.v[s][0], acc);
    }
#pragma unroll
    for (int r = 0; r < FIN_PTS / 4; ++r) ms[w][t][r * 64 + lane] = acc[r];
  }
  __syncthreads();
  for (int e = tid; e < FIN_PTS * D; e += 256) {
    const int nn = e / D, d = e % D, n = n0 + nn;
    if (n >= N) continue;
    double s = 0.0;
    for (int sp0 = 0; sp0 < S; sp0 += 4) {
      double pv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) pv[u] = part[((long)min(sp0 + u, S - 1) * N + n) * D + d];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (sp0 + u < S) s += pv[u];
    }
    const int i = (nn >> 2) * 64 + (nn & 3) * 16 + (d & 15), t = d >> 4;
    const double m = ms[0][t][i] + ms[1][t][i] + ms[2][t][i] + ms[3][t][i];
    mout[(long)n * D + d] = m;
    vout[(long)n * D + d] = sf2 + s - m * m;
  }
}

}  // namespace

extern "C" int gpx_gemm_batched(int transA, int transB, int m, int n, int k, double alpha,
                                const double *A, int lda, long strideA, const double *B, int ldb,
                                long strideB, double beta, double *C, int ldc, long strideC,
                                int batch, int splits, double *work, int tile, void *stream);
extern "C" {

long gpx_fused_bwd_workspace(int N, int M, int Q, int D, int splits, int nsplit) {
  const long MM = (long)M * M;
  long s = (long)nsplit * D * MM + (long)nsplit * MM * (Q + 1) + MM * (Q + 1);  // dBpart, LWpart, LW
  s += (long)fused_t_slots(M) * N * M + (long)fused_v_slots(M) * N * Q;  // Tpart, Vpart
  s += (long)N * M + (long)rows_finish_blocks(N, M, Q) * (M * Q + Q + 2);           // dpsi1, row finish's partials
  s += (long)N * PF_W + (long)N * M;                                          // point features, u
  return s;
}

}  // extern "C"

namespace {

// Workspace of the fused adjoint (gpx_fused_bwd_workspace doubles), carved in order.
struct FusedBwdWork {
  double *dBpart, *LWpart, *LW, *Tpart, *Vpart, *dpsi1, *rows, *un, *pf;
  FusedBwdWork(double *work, int N, int M, int Q, int D, int splits, int nsplit) {
    const long MM = (long)M * M;
    dBpart = work;
    LWpart = dBpart + (long)nsplit * D * MM;
    LW = LWpart + (long)nsplit * MM * (Q + 1);
    Tpart = LW + MM * (Q + 1);
    Vpart = Tpart + (long)fused_t_slots(M) * N * M;
    dpsi1 = Vpart + (long)fused_v_slots(M) * N * Q;
    rows = dpsi1 + (long)N * M;
    un = rows + (long)rows_finish_blocks(N, M, Q) * (M * Q + Q + 2);
    pf = un + (long)N * M;
  }
};

bool fused_bwd_args_ok(int N, int M, int Q, int D, int splits, int nsplit) {
  // Q <= FQ_MAX - 1: the [1 | d_n] contraction fills the Q+1 rows of one 16-row MFMA tile.
  // splits is an argument of an earlier form of the per-point pass, still range-checked.
  return N >= 1 && M >= 1 && M <= FM_MAX && Q >= 1 && Q <= FQ_MAX - 1 && D >= 1 && D <= 32 && splits >= 1 &&
         nsplit >= 1 && splits <= (M + 15) / 16;
}

}  // namespace

extern "C" {

// Adjoint of the moment-matched layer without materialising psi2 or dL/dpsi2:
// given dm_all = dm - 2 dv m and dv (N x D), Ahat (D x M), Bp (pair-major symmetrised
// Bhat, M x M x D) and psi1 from the forward: dBhat (D x M x M), dsf2, dell, dZ, dmx, dvx.
// dL/dpsi2 = sum_d dv_nd Bsym[d] is symmetric by construction (kernels.py:415-418).
// The work splits into three ordered parts on one `work` buffer: _points (point features,
// the adjoint kernel and the row finish: dmx and dvx, what the layer below needs), _pairs
// (the sum of its per-pair partials: dBhat and LW) and _tail (dsf2, dell, dZ).  _pairs
// and _tail may run on another stream once _points has completed there; _main is _points
// then _pairs.
int gpx_fused_mm_bwd_points(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                            const double *ls, const double *sf, const double *Ahat, const double *Bp,
                            const double *psi1, const double *dm_all, const double *dv, int splits, int nsplit,
                            double *dmx, double *dvx, double *work, void *stream) {
  if (!fused_bwd_args_ok(N, M, Q, D, splits, nsplit)) return GPX_EINVAL;
  if (!mx || !vx || !z || !ls || !sf || !Ahat || !Bp || !psi1 || !dm_all || !dv || !dmx || !dvx || !work)
    return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  FusedBwdWork W(work, N, M, Q, D, splits, nsplit);
  hipLaunchKernelGGL(fused_point_feat_kernel, dim3(gpx_cdiv(N, PF_PTS)), dim3(256), 0, st, N, M, Q, mx, vx, z, ls, W.pf,
                     W.un);
  GPX_CHECK_LAUNCH();
  // both passes in one kernel: the per-pair partials (dBpart, LWpart) are written here too,
  // and gpx_fused_mm_bwd_pairs only sums them
  const int T = (M + 15) / 16, ntiles = T * (T + 1) / 2;
  const int nchunk = ((N + nsplit - 1) / nsplit + 15) / 16 * 16;
  dim3 gm(ntiles, nsplit);
#define GPX_MERGED(DSV, KSV, GV)                                                                                \
  hipLaunchKernelGGL((fused_bwd_merged_kernel<DSV, KSV, GV>), gm, dim3(64 * MG_NW), 0, st, N, M, Q, D, z, sf, Bp, \
                     dv, (const double *)W.pf, (const double *)W.un, nsplit, nchunk, W.dBpart, W.LWpart, W.Tpart, W.Vpart)
  // KS = ceil(Q / 4) slices of the exponent, G = ceil((Q + 1) / 4) groups of [1 | z]
#define GPX_MERGED_KS(DSV)                            \
  if (Q <= 3) GPX_MERGED(DSV, 1, 1);                  \
  else if (Q == 4) GPX_MERGED(DSV, 1, 2);             \
  else if (Q <= 7) GPX_MERGED(DSV, 2, 2);             \
  else if (Q == 8) GPX_MERGED(DSV, 2, 3);             \
  else if (Q <= 11) GPX_MERGED(DSV, 3, 3);            \
  else if (Q == 12) GPX_MERGED(DSV, 3, 4);            \
  else GPX_MERGED(DSV, 4, 4);
  if (D <= 4) { GPX_MERGED_KS(1) }
  else if (D <= 8) { GPX_MERGED_KS(2) }
  else if (D <= 12) { GPX_MERGED_KS(3) }
  else if (D <= 16) { GPX_MERGED_KS(4) }
  else { GPX_MERGED_KS(8) }
#undef GPX_MERGED_KS
#undef GPX_MERGED
  GPX_CHECK_LAUNCH();
  // dpsi1 = dm_all Ahat
  int rc = gpx_gemm_batched(0, 0, N, M, D, 1.0, dm_all, D, 0, Ahat, M, 0, 0.0, W.dpsi1, M, 0, 1, 1, nullptr, 0,
                            stream);
  if (rc) return rc;
  const int kr = (Q + 3) / 4, rows_lds = (int)sizeof(double) * M * (4 * kr + 1);
#define GPX_ROWS(KRV, MJV)                                                                                    \
  hipLaunchKernelGGL((fused_rows_finish<KRV, MJV>), dim3(rows_finish_blocks(N, M, Q)), dim3(256), rows_lds, st, N, M, Q, \
                     fused_t_slots(M), fused_v_slots(M), mx, vx, z, ls, (const double *)W.Tpart,              \
                     (const double *)W.Vpart, (const double *)W.dpsi1, psi1, dmx, dvx, W.rows)
#define GPX_ROWS_MJ(KRV) \
  if (M <= 64) GPX_ROWS(KRV, 1); else if (M <= 128) GPX_ROWS(KRV, 2); else if (M <= 192) GPX_ROWS(KRV, 3); \
  else GPX_ROWS(KRV, 4);
  if (kr == 1) { GPX_ROWS_MJ(1) }
  else if (kr == 2) { GPX_ROWS_MJ(2) }
  else if (kr == 3) { GPX_ROWS_MJ(3) }
  else { GPX_ROWS_MJ(4) }
#undef GPX_ROWS_MJ
#undef GPX_ROWS
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_fused_mm_bwd_pairs(int N, int M, int Q, int D, const double *z, const double *ls, const double *sf,
                           const double *Bp, const double *dv, int splits, int nsplit, double *dBhat, double *work,
                           void *stream) {
  if (!fused_bwd_args_ok(N, M, Q, D, splits, nsplit)) return GPX_EINVAL;
  if (!z || !ls || !sf || !Bp || !dv || !dBhat || !work) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const int T = (M + 15) / 16, ntiles = T * (T + 1) / 2;
  FusedBwdWork W(work, N, M, Q, D, splits, nsplit);
  // the partials came from the kernel of the per-point part
  hipLaunchKernelGGL(fused_pairs_finish, dim3(ntiles, D + Q + 1), dim3(256), 0, st, M, Q, D, nsplit,
                     (const double *)W.dBpart, (const double *)W.LWpart, dBhat, W.LW);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_fused_mm_bwd_main(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                          const double *ls, const double *sf, const double *Ahat, const double *Bp,
                          const double *psi1, const double *dm_all, const double *dv, int splits, int nsplit,
                          double *dBhat, double *dmx, double *dvx, double *work, void *stream) {
  if (!dBhat) return GPX_EINVAL;
  const int rc = gpx_fused_mm_bwd_points(N, M, Q, D, mx, vx, z, ls, sf, Ahat, Bp, psi1, dm_all, dv, splits, nsplit,
                                         dmx, dvx, work, stream);
  if (rc) return rc;
  return gpx_fused_mm_bwd_pairs(N, M, Q, D, z, ls, sf, Bp, dv, splits, nsplit, dBhat, work, stream);
}

int gpx_fused_mm_bwd_tail(int N, int M, int Q, int D, const double *z, const double *ls, const double *sf,
                          int splits, int nsplit, double *dsf2, double *dell, double *dZ, double *work,
                          void *stream) {
  if (!fused_bwd_args_ok(N, M, Q, D, splits, nsplit)) return GPX_EINVAL;
  if (!z || !ls || !sf || !dsf2 || !dell || !dZ || !work) return GPX_EINVAL;
  FusedBwdWork W(work, N, M, Q, D, splits, nsplit);
  hipLaunchKernelGGL(fused_tail_kernel, dim3(M + 1), dim3(256), 0, (hipStream_t)stream, M, Q, rows_finish_blocks(N, M, Q),
                     z, ls, sf, (const double *)W.LW, (const double *)W.rows, dsf2, dell, dZ);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_fused_mm_bwd(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                     const double *ls, const double *sf, const double *Ahat, const double *Bp,
                     const double *psi1, const double *dm_all, const double *dv, int splits, int nsplit,
                     double *dBhat, double *dsf2, double *dell, double *dZ, double *dmx, double *dvx,
                     double *work, void *stream) {
  if (!dsf2 || !dell || !dZ) return GPX_EINVAL;
  int rc = gpx_fused_mm_bwd_main(N, M, Q, D, mx, vx, z, ls, sf, Ahat, Bp, psi1, dm_all, dv, splits, nsplit, dBhat,
                                 dmx, dvx, work, stream);
  if (rc) return rc;
  return gpx_fused_mm_bwd_tail(N, M, Q, D, z, ls, sf, splits, nsplit, dsf2, dell, dZ, work, stream);
}

}  // extern "C"

extern "C" {


// Symmetrised Bhat in pair-major layout: out[a, b, d] = (B[d,a,b] + B[d,b,a]) / 2.
int gpx_sym_pairmajor(int D, int M, const double *B, double *out, void *stream) {
  if (D < 1 || M < 1 || !B || !out || B == out) return GPX_EINVAL;
  const long n = (long)D * M * M;
  hipLaunchKernelGGL(sym_pairmajor_kernel, dim3(gpx_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, D, M, B, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

long gpx_fused_fwd_workspace(int N, int M, int D, int splits) { return (long)splits * N * D + (long)M * M; }

// Moment-matched layer forward without materialising psi2:
// psi1 (N x M), mout = psi1 Ahat^T, vout = sf2 + <Bsym[d], psi2_n> - mout^2 (N x D).
// Bp is the symmetrised Bhat in pair-major layout (gpx_sym_pairmajor); `splits`
// spreads the pair tiles over grid.y and `nsub` (1, 2 or 4) sets 16*nsub points per block.
static int fused_fwd_check(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                           const double *ls, const double *sf, const double *Ahat, const double *Bp, int splits,
                           int nsub, const double *psi1, const double *mout, const double *vout) {
  if (N < 1 || M < 1 || M > FM_MAX || Q < 1 || Q > FQ_MAX || D < 1 || D > 32 || splits < 1)
    return GPX_EINVAL;
  if (nsub != 1 && nsub != 2 && nsub != 4) return GPX_EINVAL;
  if (!mx || !vx || !z || !ls || !sf || !Ahat || !Bp || !psi1 || !mout || !vout) return GPX_EINVAL;
  const int T = (M + 15) / 16, ntiles = T * (T + 1) / 2;
  if (splits > ntiles) return GPX_EINVAL;
  return GPX_OK;
}

// The launches of gpx_fused_mm_fwd over a checked argument set and a workspace of
// gpx_fused_fwd_workspace(N, M, D, splits) doubles.
static int fused_fwd_launch(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                            const double *ls, const double *sf, const double *Ahat, const double *Bp, int splits,
                            int nsub, double *psi1, double *mout, double *vout, double *work, hipStream_t st) {
  // fewer points per workgroup where their u would not fit the LDS
  const int ks = (Q + 3) / 4;
  while (nsub > 1 && fwd_lds(M, D, ks, nsub) * sizeof(double) > kFwdLds) nsub /= 2;
  const size_t lds = fwd_lds(M, D, ks, nsub) * sizeof(double);
  dim3 grid(split_grid(gpx_cdiv(N, 16 * nsub), splits));
#define GPX_FWD1(DBV, NS, KSV)                                                                                   \
  hipLaunchKernelGGL((fused_fwd_kernel<DBV, NS, KSV>), grid, dim3(256), lds, st, N, M, Q, D, mx, vx, z, ls, sf, Bp, \
                     splits, work)
#define GPX_FWD(DBV, NS)                                                    \
  do {                                                                      \
    if (ks == 1) GPX_FWD1(DBV, NS, 1); else if (ks == 2) GPX_FWD1(DBV, NS, 2); \
    else if (ks == 3) GPX_FWD1(DBV, NS, 3); else GPX_FWD1(DBV, NS, 4);       \
  } while (0)
  if (D <= 4) {
    if (nsub == 1) GPX_FWD(0, 1); else if (nsub == 2) GPX_FWD(0, 2); else GPX_FWD(0, 4);
  } else if (D <= 16) {
    if (nsub == 1) GPX_FWD(1, 1); else if (nsub == 2) GPX_FWD(1, 2); else GPX_FWD(1, 4);
  } else {
    if (nsub == 1) GPX_FWD(2, 1); else if (nsub == 2) GPX_FWD(2, 2); else GPX_FWD(2, 4);
  }
#undef GPX_FWD
#undef GPX_FWD1
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(fused_fwd_finish, dim3(gpx_cdiv(N, FIN_PTS)), dim3(256), 0, st, N, M, Q, D, mx, vx, z, ls, sf,
                     Ahat, (const double *)work, splits, psi1, mout, vout);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_fused_mm_fwd(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                     const double *ls, const double *sf, const double *Ahat, const double *Bp,
                     int splits, int nsub, double *psi1, double *mout, double *vout, double *work,
                     void *stream) {
  const int rc = fused_fwd_check(N, M, Q, D, mx, vx, z, ls, sf, Ahat, Bp, splits, nsub, psi1, mout, vout);
  if (rc != GPX_OK) return rc;
  if (!work) return GPX_EINVAL;
  return fused_fwd_launch(N, M, Q, D, mx, vx, z, ls, sf, Ahat, Bp, splits, nsub, psi1, mout, vout, work,
                          (hipStream_t)stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Allocation-free forward.  The workspace of gpx_fused_mm_fwd (per-split partial sums
// and M x M spare doubles) lives in a file-scope device array instead of caller
// memory.  Each GPU holds its own copy of the array from module load to process exit;
// host code never passes the array's name to a kernel (in host code that name is a
// host-side stand-in), only the device address hipGetSymbolAddress returns for the
// current device, looked up once per device and kept.
// ---------------------------------------------------------------------------
namespace {

constexpr long kNoAllocScratch = 4L << 20;  // doubles (32 MiB)
__device__ __align__(256) double scratch[kNoAllocScratch];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (NULL on failure).
double *scratch_on_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    g_scratch_ptr[dev] = static_cast<double *>(p);
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" {

long gpx_fused_fwd_noalloc_max(void) { return kNoAllocScratch; }

int gpx_fused_mm_fwd_noalloc(int N, int M, int Q, int D, const double *mx, const double *vx, const double *z,
                             const double *ls, const double *sf, const double *Ahat, const double *Bp, int splits,
                             int nsub, double *psi1, double *mout, double *vout, void *stream) {
  const int rc = fused_fwd_check(N, M, Q, D, mx, vx, z, ls, sf, Ahat, Bp, splits, nsub, psi1, mout, vout);
  if (rc != GPX_OK) return rc;
  if (gpx_fused_fwd_workspace(N, M, D, splits) > kNoAllocScratch) return GPX_ETOOBIG;
  double *work = scratch_on_current_device();
  if (!work) return GPX_EHIP;
  return fused_fwd_launch(N, M, Q, D, mx, vx, z, ls, sf, Ahat, Bp, splits, nsub, psi1, mout, vout, work,
                          (hipStream_t)stream);
}

}  // extern "C"
