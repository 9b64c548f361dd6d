// SE kernel matrices, their adjoints, and the small per-layer / likelihood kernels of
// the AEP objective.  All arrays are row-major FP64 device memory; log
// hyper-parameters (ls, sf, sn, R) are read from the device so no host sync is needed.
#include "gpx_frag.h"

#include <algorithm>

namespace {

// ---------------------------------------------------------------------------
// SE kernel: compute_kernel (kernels.py:10-22), K = sf2 exp(-sum_q (x-z)^2 / (2 l_q))
// ---------------------------------------------------------------------------
// Q > 16 (any Q): one thread per entry.
__global__ void se_any_kernel(int N, int M, int Q, const double *__restrict__ x, int ldx,
                              const double *__restrict__ z, const double *__restrict__ ls,
                              const double *__restrict__ sf, double jitter, double *__restrict__ K) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= (long)N * M) return;
  const int n = (int)(e / M), m = (int)(e % M);
  double r2 = 0.0;
  for (int q = 0; q < Q; ++q) {
    const double d = x[(long)n * ldx + q] - z[m * Q + q];
    r2 += d * d / exp(2.0 * ls[q]);
  }
  double k = exp(2.0 * sf[0]) * exp(-0.5 * r2);
  if (n == m) k += jitter;
  K[e] = k;
}

// Q <= QC: a block takes CB columns (16, 32 or 64, as M fills them) by RPT 256 / CB rows, RPT a thread.
// x, 1/l and sf2 are formed once per block, a thread's z row stays in registers.  Bound by its exps and
// its writes (N = 20000, M = 200, Q = 8: 58 -> 19 us; with the lengthscales' exps and divisions per
// entry it was bound by those).  Four rows a thread; one where four would make few blocks: such a
// launch is as long as one thread's entries (us, one : four, 64 columns: 50 x 50, Q = 2 3.2 : 3.8; 256 x
// 256, Q = 10 (64 blocks) 3.4 : 4.5; 3000 x 64, Q = 3 (188) 3.9 : 4.2, Q = 8 4.4 : 4.4; 2000 x 128, Q = 8 (250) 5.0 :
// 4.6; 4000 x 128, Q = 4 (500) 4.7 : 4.7; 4000 x 32, Q = 16 (125) 6.5 : 5.2; 2500 x 64, Q = 16 (157) 8.0 : 5.7).
template <int QC, int RPT, int CB>
__global__ __launch_bounds__(256) void se_kernel(int N, int M, int Q, const double *__restrict__ x, int ldx,
                                                 const double *__restrict__ z, const double *__restrict__ ls,
                                                 const double *__restrict__ sf, double jitter,
                                                 double *__restrict__ K) {
  constexpr int step = 256 / CB, rows = RPT * step;
  __shared__ double xs[rows][QC], il[QC], s2;
  const int tid = threadIdx.x, n0 = blockIdx.x * rows, m = blockIdx.y * CB + tid % CB, i0 = tid / CB;
  if (tid < QC) il[tid] = tid < Q ? exp(-2.0 * ls[tid]) : 0.0;
  if (tid == 255) s2 = exp(2.0 * sf[0]);
  for (int e = tid; e < rows * QC; e += 256) {
    const int i = e / QC, q = e % QC;
    xs[i][q] = q < Q ? x[(long)min(n0 + i, N - 1) * ldx + q] : 0.0;
  }
  double zr[QC];
#pragma unroll
  for (int q = 0; q < QC; ++q) zr[q] = q < Q ? z[min(m, M - 1) * Q + q] : 0.0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    const int i = i0 + step * u, n = n0 + i;
    double r2 = 0.0;
#pragma unroll
    for (int q = 0; q < QC; ++q) {
      const double d = xs[i][q] - zr[q];
      r2 = fma(d * il[q], d, r2);
    }
    double k = s2 * exp(-0.5 * r2);
    if (n == m) k += jitter;
    if (n < N && m < M) K[(long)n * M + m] = k;
  }
}

// kfucompDer (kernels.py:381-399) with L = dK * K.  Pass 1: block b takes the rows b G + g,
// b G + g + nblk G, ...; thread (g, m) (m < MP, the columns rounded up to 64, 128 or 256;
// G = 256 / MP row groups) keeps colsum_m, sum_n L x_nq and sum_n L (z_mq - x_nq)^2 in
// registers (QC >= Q), the groups are added in order through LDS, and the W = 2Q + 1
// sums go to part[b][w][m].  Bound by reading dK and K once; partials of 16-row slabs summed
// by 14 workgroups were most of the adjoint before (three passes at N = 20000, M = 200, Q = 8
// 104 -> 38 us; N = 1000, M = 100, Q = 10 17 -> 18 us).
// REG: dK is formed here, dK_nm = sum_d dm_nd A_dm + 2 dv_nd T_dnm (the propagation's adjoint at
// deterministic inputs), which a product, a weighted sum over T and this pass wrote and read three
// times; and sum_nd dv, one value per block, goes to part[b][2Q + 1][0].
struct KfuReg {
  int D;
  const double *dm, *dv, *A, *T;
};

template <int QC, bool REG>
__global__ __launch_bounds__(256) void kfu_bwd_partial(int N, int M, int Q, int MP, const double *__restrict__ dK,
                                                       KfuReg reg, const double *__restrict__ K,
                                                       const double *__restrict__ x,
                                                       const double *__restrict__ z,
                                                       double *__restrict__ part) {
  __shared__ double red[2 * QC + 1][256];
  __shared__ double sdv[4];
  // g is uniform over a wave (MP a multiple of 64): its x rows are scalar loads
  const int tid = threadIdx.x, m = tid % MP, g = __builtin_amdgcn_readfirstlane(tid / MP), G = 256 / MP,
            mc = min(m, M - 1);
  double zr[QC], lx[QC], ld2[QC], cs = 0.0, vsum = 0.0;
#pragma unroll
  for (int q = 0; q < QC; ++q) {
    zr[q] = q < Q ? z[mc * Q + q] : 0.0;
    lx[q] = ld2[q] = 0.0;
  }
  const int step = gridDim.x * G;
  // four rows' loads in flight together (rows past the end clamped, their L zeroed)
  for (int n = blockIdx.x * G + g; n < N; n += 4 * step) {
    double L[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long o = (long)min((long)n + (long)u * step, N - 1L) * M + mc;
      if constexpr (REG) L[u] = 0.0; else L[u] = dK[o] * K[o];
    }
    if constexpr (REG) {
      const int D = reg.D;
#pragma unroll 2
      for (int d = 0; d < D; ++d) {
        const double a = reg.A[(long)d * M + mc];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const long rr = (long)n + (long)u * step, r = min(rr, N - 1L);
          const double vv = reg.dv[r * D + d];
          L[u] = fma(2.0 * vv, reg.T[((long)d * N + r) * M + mc], fma(reg.dm[r * D + d], a, L[u]));
          if (rr < N) vsum += vv;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) L[u] *= K[(long)min((long)n + (long)u * step, N - 1L) * M + mc];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long r = (long)n + (long)u * step;
      const double Lu = r < N ? L[u] : 0.0;
      const double *xr = x + min(r, N - 1L) * Q;
      cs += Lu;
#pragma unroll
      for (int q = 0; q < QC; ++q) {
        const double xv = xr[min(q, Q - 1)], d = zr[q] - xv;  // q >= Q: never stored
        lx[q] = fma(Lu, xv, lx[q]);
        ld2[q] = fma(Lu * d, d, ld2[q]);
      }
    }
  }
  red[0][tid] = cs;
#pragma unroll
  for (int q = 0; q < QC; ++q) {
    red[1 + q][tid] = lx[q];
    red[1 + QC + q][tid] = ld2[q];
  }
  if (REG && m == 0) sdv[g] = vsum;  // the same in every column of the group
  __syncthreads();
  const int W = 2 * Q + 1, rows = REG ? W + 1 : W;
  for (int e = tid; e < W * M; e += 256) {
    const int w = e / M, c = e % M, r = w <= Q ? w : w - Q + QC;
    double s = red[r][c];
    for (int h = 1; h < G; ++h) s += red[r][h * MP + c];
    part[((long)blockIdx.x * rows + w) * M + c] = s;
  }
  if (REG && tid == 0) {
    double s = sdv[0];
    for (int h = 1; h < G; ++h) s += sdv[h];
    part[((long)blockIdx.x * rows + W) * M] = s;
  }
}

// dx_nq = sum_m L_nm (z_mq - x_nq) / l_q of row n by one wave: lane (g, c) takes q = g + 4 k (k < KR) and
// m = c, c + 16, ..., so the row's Q sums are KR sums over 16 lanes.  z: LDS, rows of zld.
template <int KR>
__device__ __forceinline__ void kfu_dx_row(long n, int lane, int M, int Q, const double *dK, const double *K,
                                           const double *x, const double *z, int zld, const double *ls, double *dx) {
  const int g = lane >> 4, c = lane & 15;
  double xv[KR], s[KR];
#pragma unroll
  for (int k = 0; k < KR; ++k) {
    xv[k] = x[n * Q + min(g + 4 * k, Q - 1)];
    s[k] = 0.0;
  }
#pragma unroll 2
  for (int m0 = 0; m0 < M; m0 += 16) {
    const int mc = min(m0 + c, M - 1);
    const double L = dK[n * M + mc] * K[n * M + mc] * (m0 + c < M ? 1.0 : 0.0);
#pragma unroll
    for (int k = 0; k < KR; ++k) s[k] = fma(L, z[mc * zld + min(g + 4 * k, Q - 1)] - xv[k], s[k]);
  }
#pragma unroll
  for (int k = 0; k < KR; ++k) {
    const int q = g + 4 * k;
    const double t = gpx_row_sum(s[k]);
    if (c == 0 && q < Q) dx[n * Q + q] = t / exp(2.0 * ls[q]);
  }
}

// Pass 2: red[w][m] = sum over the blocks of part[b][w][m]: 64 columns by 16 groups of blocks
// (loads eight at a time), the groups added in order.  KR > 0: the workgroups past the first `sums`
// form dx, a wave to a row, with z in LDS (M rows of Q | 1).  Whole adjoint with dx, us: N = 1000, M = 100,
// Q = 10 16.4 (18.3 with dx in the first pass, 19.5 in a launch of its own with a wave sum over m for
// each q), 20000, 200, 16 88 (135, 195; 97 with two rows a wave).
template <int KR>
__global__ __launch_bounds__(1024) void kfu_bwd_final(int nblk, int M, int W, int sums, const double *__restrict__ part,
                                                      double *__restrict__ red, int N, int Q,
                                                      const double *__restrict__ dK, const double *__restrict__ K,
                                                      const double *__restrict__ x, const double *__restrict__ z,
                                                      const double *__restrict__ ls, double *__restrict__ dx) {
  __shared__ double sm[16][64];
  extern __shared__ double zs[];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
  if constexpr (KR > 0) {
    if ((int)blockIdx.x >= sums) {  // uniform over the workgroup
      const int zld = Q | 1;
      const long n = ((long)blockIdx.x - sums) * 16 + g;
      for (int e = threadIdx.x; e < M * Q; e += 1024) zs[e / Q * zld + e % Q] = z[e];
      __syncthreads();
      if (n < N) kfu_dx_row<KR>(n, c, M, Q, dK, K, x, zs, zld, ls, dx);
      return;
    }
  }
  const int cb = (M + 63) >> 6, m = (int)blockIdx.x % cb * 64 + c, w = (int)blockIdx.x / cb;
  const double *P = part + (long)w * M + min(m, M - 1);
  const long bs = (long)W * M;
  double s = 0.0;
#pragma unroll 8
  for (int b = g; b < nblk; b += 16) s += P[b * bs];
  sm[g][c] = s;
  __syncthreads();
  if (g == 0 && m < M) {
    double t = sm[0][c];
#pragma unroll
    for (int h = 1; h < 16; ++h) t += sm[h][c];
    red[(long)w * M + m] = t;
  }
}

// Pass 3, one wave per output j <= Q, lanes over m and a fixed-order wave reduction:
// dsf2 = sum_m colsum_m / sf2, dell_q = sum_m Ld2_mq / ell^3, and
// dZ_mq = -(z_mq colsum_m - Lx_mq) / l_q.  extra (may be NULL) is added to dsf2.
__global__ __launch_bounds__(64) void kfu_bwd_scalars(int M, int Q, const double *__restrict__ red,
                                                      const double *__restrict__ extra,
                                                      const double *__restrict__ z,
                                                      const double *__restrict__ ls,
                                                      const double *__restrict__ sf, double *__restrict__ dsf2,
                                                      double *__restrict__ dell, double *__restrict__ dZ) {
  const int j = blockIdx.x, lane = threadIdx.x;
  const double l = j ? exp(2.0 * ls[j - 1]) : 1.0;
  double s = 0.0;
  for (int m = lane; m < M; m += 64) {
    const double cs = red[m];
    s += j == 0 ? cs : red[(long)(Q + j) * M + m];
    if (j) dZ[m * Q + j - 1] = -(z[m * Q + j - 1] * cs - red[(long)j * M + m]) / l;
  }
  s = gpx_wave_sum(s);
  if (lane == 0) {
    if (j == 0)
      dsf2[0] = extra ? s / exp(2.0 * sf[0]) + extra[0] : s / exp(2.0 * sf[0]);
    else
      dell[j - 1] = s / exp(3.0 * ls[j - 1]);
  }
}

// d_trace_MKzz_dhypers (kernels.py:447-475) with Kzz = SE(z, z) (no jitter):
//   gsf = sum_ab M_ab K_ab, gls_q = sum_ab M_ab K_ab (z_aq - z_bq)^2 / (2 l_q),
//   gz_aq = -sum_b (M_ab + M_ba) K_ab (z_aq - z_bq) / l_q.
// One wave per row a (four per workgroup), its lanes over b; part[a] = [gsf_a, gls_a (Q)].
// Z (q-major, so lanes b read consecutive words) and 1/l_q are staged in LDS once per
// workgroup; QT = Q fixes the per-lane arrays.
template <int QT>
__global__ __launch_bounds__(256) void dtrace_kernel(int M, const double *__restrict__ Mm,
                                                     const double *__restrict__ z,
                                                     const double *__restrict__ ls,
                                                     const double *__restrict__ sf, const double *dz0,
                                                     double *gz, double *__restrict__ part) {
  __shared__ double zs[QT][256];
  __shared__ double ils[QT];
  const int tid = threadIdx.x, lane = tid & 63, a = blockIdx.x * 4 + (tid >> 6);
  for (int e = tid; e < M * QT; e += 256) zs[e % QT][e / QT] = z[e];
  if (tid < QT) ils[tid] = 1.0 / exp(2.0 * ls[tid]);
  __syncthreads();
  if (a >= M) return;  // whole waves, after the only barrier
  const double sf2 = exp(2.0 * sf[0]);
  double il[QT], za[QT], gl[QT], gzq[QT];
#pragma unroll
  for (int q = 0; q < QT; ++q) {
    il[q] = ils[q];
    za[q] = zs[q][a];
    gl[q] = gzq[q] = 0.0;
  }
  double g0 = 0.0;
  for (int b = lane; b < M; b += 64) {
    double r2 = 0.0, d[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) {
      d[q] = za[q] - zs[q][b];
      r2 += d[q] * d[q] * il[q];
    }
    const double K = sf2 * exp(-0.5 * r2);
    const double mab = Mm[(long)a * M + b], mba = Mm[(long)b * M + a];
    g0 += mab * K;
#pragma unroll
    for (int q = 0; q < QT; ++q) {
      gl[q] += 0.5 * mab * K * d[q] * d[q] * il[q];
      gzq[q] += (mab + mba) * K * d[q];
    }
  }
  g0 = gpx_wave_sum(g0);
#pragma unroll
  for (int q = 0; q < QT; ++q) {
    gl[q] = gpx_wave_sum(gl[q]);
    gzq[q] = gpx_wave_sum(gzq[q]);
  }
  if (lane == 0) part[(long)a * (QT + 1)] = g0;
#pragma unroll
  for (int q = 0; q < QT; ++q)
    if (lane == q) {
      part[(long)a * (QT + 1) + 1 + q] = gl[q];
      gz[a * QT + q] = dz0 ? dz0[a * QT + q] - gzq[q] * il[q] : -gzq[q] * il[q];
    }
}

// One wave per output column j <= Q: lanes stride over the M rows, then a fixed-order
// wave reduction (a single thread per column summing M dependent loads was 16 us).
__global__ __launch_bounds__(64) void dtrace_final(int M, int Q, const double *__restrict__ part,
                                                   double *__restrict__ gsf, double *__restrict__ gls) {
  const int j = blockIdx.x, lane = threadIdx.x;
  double s = 0.0;
  for (int a = lane; a < M; a += 64) s += part[(long)a * (Q + 1) + j];
  s = gpx_wave_sum(s);
  if (lane == 0) {
    if (j == 0) gsf[0] = s;
    else gls[j - 1] = s;
  }
}

// dtrace_final with the chain rule of the log hyper-parameters (hyper_kernel) applied.
__global__ __launch_bounds__(64) void kuu_tail_kernel(int M, int Q, const double *__restrict__ part,
                                                      const double *__restrict__ ls, const double *__restrict__ sf,
                                                      const double *__restrict__ dell,
                                                      const double *__restrict__ dsf2,
                                                      const double *__restrict__ sumdv, double *__restrict__ dls,
                                                      double *__restrict__ dsf) {
  const int j = blockIdx.x, lane = threadIdx.x;
  double s = 0.0;
  for (int a = lane; a < M; a += 64) s += part[(long)a * (Q + 1) + j];
  s = gpx_wave_sum(s);
  if (lane != 0) return;
  if (j == 0) dsf[0] = 2.0 * exp(2.0 * sf[0]) * (sumdv ? dsf2[0] + sumdv[0] : dsf2[0]) + 2.0 * s;
  else dls[j - 1] = dell[j - 1] * exp(ls[j - 1]) + 2.0 * s;
}

// mu_b = s_b S_b t_b and P_b = S_b + mu_b mu_b^T.  M <= 64: one launch, a workgroup per matrix, whose waves
// keep their rows in registers between the two.  Above, the means (a wave per row) and then P (a thread
// per element): all of it is latency, and rows read again, or several rows a wave, cost more than the
// launch (us: M = 50, 2 matrices 4.2, two launches 5.4; M = 100, 10 6.0, one launch that formed the means
// again in each workgroup 8.5; 256, 4 6.0, four rows a wave in both 9.6).
__global__ __launch_bounds__(1024) void moments_kernel(int D, int M, const double *__restrict__ S,
                                                       const double *__restrict__ theta, double s0, double s1,
                                                       double *__restrict__ mu, double *__restrict__ P) {
  __shared__ double m[64];
  const int b = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = min(lane, M - 1);
  const double *Sb = S + (long)b * M * M;
  const double t = lane < M ? theta[(long)(b % D) * M + c] : 0.0, scale = b < D ? s0 : s1;
  double v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = Sb[(long)min(w + 16 * u, M - 1) * M + c];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const double s = gpx_wave_sum(lane < M ? v[u] * t : 0.0);
    if (lane == 0 && w + 16 * u < M) m[w + 16 * u] = scale * s;
  }
  __syncthreads();
  if (lane >= M) return;
  if (w == 0) mu[(long)b * M + lane] = m[lane];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = w + 16 * u;
    if (i < M) P[(long)b * M * M + (long)i * M + lane] = m[i] * m[lane] + v[u];
  }
}

__global__ __launch_bounds__(256) void mean_kernel(int D, int M, const double *__restrict__ S,
                                                   const double *__restrict__ theta, double s0, double s1,
                                                   double *__restrict__ mu) {
  const int b = blockIdx.x, lane = threadIdx.x & 63, i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= M) return;  // whole waves, no barriers
  const double *row = S + ((long)b * M + i) * M, *t = theta + (long)(b % D) * M;
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = lane + 64 * j;
    const double v = row[min(c, M - 1)] * t[min(c, M - 1)];
    acc += c < M ? v : 0.0;
  }
  acc = gpx_wave_sum(acc);
  if (lane == 0) mu[(long)b * M + i] = (b < D ? s0 : s1) * acc;
}

__global__ __launch_bounds__(256) void second_kernel(int M, const double *__restrict__ S,
                                                     const double *__restrict__ mu, double *__restrict__ P) {
  const int b = blockIdx.x, e = blockIdx.y * 256 + threadIdx.x;
  if (e >= M * M) return;
  const double *m = mu + (long)b * M;
  const long o = (long)b * M * M + e;
  P[o] = m[e / M] * m[e % M] + S[o];
}

// One block per column, threads stride over the rows (fixed-order block reduction).
__global__ __launch_bounds__(256) void colsum_tall_kernel(int rows, int cols, const double *__restrict__ P,
                                                          double alpha, double beta, double *__restrict__ out) {
  __shared__ double red[16];
  const int j = blockIdx.x;
  double s = 0.0;
#pragma unroll 8
  for (long i = threadIdx.x; i < rows; i += 256) s += P[i * cols + j];
  s = gpx_block_sum(s, red);
  if (threadIdx.x == 0) out[j] = (beta == 0.0) ? alpha * s : alpha * s + beta * out[j];
}

// Stage 1 of the two-stage column sum: block (j, c) sums rows [c*chunk, (c+1)*chunk) of
// column j into part[c * cols + j] (strided loads, fixed-order block reduction).
__global__ __launch_bounds__(256) void colsum_chunk_kernel(int rows, int cols, int chunk,
                                                           const double *__restrict__ P,
                                                           double *__restrict__ part) {
  __shared__ double red[16];
  const int j = blockIdx.x, c = blockIdx.y;
  const long r0 = (long)c * chunk, r1 = min((long)rows, r0 + chunk);
  double s0 = 0.0, s1 = 0.0;
  long i = r0 + threadIdx.x;
  for (; i + 256 < r1; i += 512) {
    s0 += P[i * cols + j];
    s1 += P[(i + 256) * cols + j];
  }
  if (i < r1) s0 += P[i * cols + j];
  const double s = gpx_block_sum(s0 + s1, red);
  if (threadIdx.x == 0) part[(long)c * cols + j] = s;
}

__global__ void colsum_kernel(int rows, int cols, const double *__restrict__ P, double alpha,
                              double beta, double *__restrict__ out) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= cols) return;
  double s = 0.0;
  // unrolled: eight loads in flight ahead of the (same-order) adds
#pragma unroll 8
  for (int i = 0; i < rows; ++i) s += P[(long)i * cols + j];
  out[j] = (beta == 0.0) ? alpha * s : alpha * s + beta * out[j];
}

// ---------------------------------------------------------------------------
// q(u) parameter plumbing (base_models.py:645-653; aep_models.py:267-280)
// ---------------------------------------------------------------------------
__device__ __forceinline__ long triu_index(int M, int i, int j) {
  return (long)i * M - (long)i * (i - 1) / 2 + (j - i);
}

__global__ void eta_to_R_kernel(int D, int M, const double *__restrict__ eta, double *__restrict__ R) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const long MM = (long)M * M;
  if (e >= D * MM) return;
  const int d = (int)(e / MM), i = (int)((e % MM) / M), j = (int)(e % M);
  double v = 0.0;
  if (j >= i) {
    const double t = eta[(long)d * (M * (M + 1) / 2) + triu_index(M, i, j)];
    v = (i == j) ? exp(t) : t;
  }
  R[e] = v;
}

// out[d, triu(i,j)] = (sum_{k>=i} R_ik (G_kj + G_jk)) * (i == j ? R_ii : 1)
// One workgroup per upper 16 x 16 output tile (I, J >= I) of one d: the product R (G + G^T) over
// k >= 16 I (R is upper triangular) on the FP64 matrix cores, operands straight from global
// memory, each wave every fourth group of 8 k and two groups in flight; the waves' sums are added
// in wave order.  Bound by the load latency of a wave's share (a wave per tile walked all of k:
// D = 32, M = 128 17 -> 10 us, D = 2, M = 256 18 -> 5.7, D = 1, M = 50 5.2 -> 2.9).
__global__ __launch_bounds__(256) void pack_dR_kernel(int D, int M, const double *__restrict__ R,
                                                      const double *__restrict__ G, double *__restrict__ out) {
  __shared__ double red[4][256];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane >> 4,
            lc = lane & 15;
  const int MT = (M + 15) / 16;
  int t = blockIdx.x, I = 0;
  while (t >= MT - I) {
    t -= MT - I;
    ++I;
  }
  const int J = I + t, d = blockIdx.y, k0 = 16 * I;
  const double *Rd = R + (long)d * M * M, *Gd = G + (long)d * M * M;
  const GpxOperand<1, true> oa(Rd, M, k0, M, lane), oc(Gd, M, 16 * J, M, lane);
  const GpxOperand<1, false> ob(Gd, M, 16 * J, M, lane);
  gpx_d4 acc = {0.0, 0.0, 0.0, 0.0};
  GpxFrag<1> a[2], g[2], h[2];
  auto mul = [&](int u) {
#pragma unroll
    for (int s = 0; s < 2; ++s) acc = gpx_mfma16(a[u].v[s][0], g[u].v[s][0] + h[u].v[s][0], acc);
  };
  const int groups = (M - k0) >> 3, mine = (groups - w + 3) / 4, kr = (M - k0) & 7;
  if (mine > 0) {
    auto load = [&](int u, int t) {
      const int k = k0 + 8 * (w + 4 * min(t, mine - 1));
      oa.load(a[u], k);
      ob.load(g[u], k);
      oc.load(h[u], k);
    };
    load(0, 0);
    int t = 0;
    for (; t + 2 <= mine; t += 2) {
      load(1, t + 1);
      mul(0);
      load(0, t + 2);
      mul(1);
    }
    if (t < mine) mul(0);
  }
  if (kr && w == groups % 4) {
    oa.load_tail(a[0], k0 + 8 * groups, kr, lane);
    ob.load_tail(g[0], k0 + 8 * groups, kr, lane);
    oc.load_tail(h[0], k0 + 8 * groups, kr, lane);
    mul(0);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[w][r * 64 + lane] = acc[r];
  __syncthreads();
  const int ii = k0 + lr + 4 * w, jj = J * 16 + lc;  // wave w finishes register w
  if (ii >= M || jj >= M || jj < ii) return;
  const int e = w * 64 + lane;
  const double v = red[0][e] + red[1][e] + red[2][e] + red[3][e];
  const long rowoff = (long)ii * M - (long)ii * (ii - 1) / 2;
  out[(long)d * ((long)M * (M + 1) / 2) + rowoff + (jj - ii)] = ii == jj ? v * Rd[(long)ii * M + ii] : v;
}

__global__ void lincomb_kernel(long n, double a, const double *__restrict__ x, long nx, double b,
                               const double *__restrict__ y, long ny, double c,
                               const double *__restrict__ w, long nw, double *__restrict__ out) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    double v = a * x[i % nx];
    if (y) v += b * y[i % ny];
    if (w) v += c * w[i % nw];
    out[i] = v;
  }
}

__global__ void sym_kernel(int batch, int M, double a, const double *__restrict__ X, double *__restrict__ out) {
  const long MM = (long)M * M;
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= batch * MM) return;
  const long base = (e / MM) * MM;
  const int i = (int)((e % MM) / M), j = (int)(e % M);
  out[e] = a * (X[base + (long)i * M + j] + X[base + (long)j * M + i]);
}

// v[n,d] = sf2 + sum_a T[d][n][a] kfu[n][a]   (aep_models.py:155-157)
// One wave per (n, d), its lanes over a (coalesced rows of T and kfu).
__global__ __launch_bounds__(256) void det_var_kernel(int N, int D, int M, const double *__restrict__ T,
                                                      const double *__restrict__ kfu, const double *__restrict__ sf,
                                                      double *__restrict__ v) {
  const long e = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (e >= (long)N * D) return;
  const int n = (int)(e / D), d = (int)(e % D);
  const double *t = T + ((long)d * N + n) * M, *k = kfu + (long)n * M;
  double s = 0.0;
  for (int a = lane; a < M; a += 64) s += t[a] * k[a];
  s = gpx_wave_sum(s);
  if (lane == 0) v[e] = exp(2.0 * sf[0]) + s;
}

// v = sf2 + Bpsi2 - m^2   (aep_models.py:196-198)
__global__ void mm_var_kernel(long n, const double *__restrict__ m, const double *__restrict__ Bp,
                              const double *__restrict__ sf, double *__restrict__ v) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= n) return;
  v[e] = exp(2.0 * sf[0]) + Bp[e] - m[e] * m[e];
}

// out[b] = sum_i x[b][i] y[b][i]
__global__ void batched_dot_kernel(int batch, int n, const double *__restrict__ x,
                                   const double *__restrict__ y, double *__restrict__ out) {
  __shared__ double red[16];
  const int b = blockIdx.x;
  double s = 0.0;
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += blockDim.x) s += x[(long)b * n + i] * y[(long)b * n + i];
  s = gpx_block_sum(s, red);
  if (threadIdx.x == 0) out[b] = s;
}

// ---------------------------------------------------------------------------
// Gauss_Layer.compute_log_Z + backprop_grads (lik_layers.py:104-181), 2-D branch.
// scal[0] = logZ (with the alpha constant), scal[1] = dsn (scaled).
// dm/dv outputs are scaled by `scale`; dmall = dm - 2 dv m when requested.
// ---------------------------------------------------------------------------
// Bound by the latency of an element's log and division: as few elements per thread as 64 blocks
// (their partials) allow (131072 elements 11.6 -> 6.1 us, 1000 7.3 -> 4.4).
__global__ __launch_bounds__(1024) void gauss_tilted_kernel(int B, int D, const double *__restrict__ m,
                                                           const double *__restrict__ v,
                                                           const double *__restrict__ y,
                                                           const double *__restrict__ sn, double alpha,
                                                           double scale, double *__restrict__ dm,
                                                           double *__restrict__ dv,
                                                           double *__restrict__ dmall,
                                                           double *__restrict__ part) {
  __shared__ double red[16];
  const double sn2 = exp(2.0 * sn[0]);
  const double two_pi = 6.283185307179586;
  double lz = 0.0, sdv = 0.0;
  const long n = (long)B * D;
  const double sa = sn2 / alpha;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    // two divisions: r (1/vt) would be off by half an ulp more than r / vt
    const double vt = v[e] + sa, iv = 1.0 / vt;
    const double r = y[e] - m[e], gm = r / vt;
    lz += -0.5 * (log(two_pi * vt) + r * gm);
    const double gv = 0.5 * (gm * gm - iv);
    sdv += gv;
    dm[e] = scale * gm;
    dv[e] = scale * gv;
    if (dmall) dmall[e] = scale * gm - 2.0 * scale * gv * m[e];
  }
  lz = gpx_block_sum(lz, red);
  sdv = gpx_block_sum(sdv, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = lz;
    part[2 * blockIdx.x + 1] = sdv;
  }
}

// One wave, lane b holding block b's partials (nblk <= 64), then fixed-order wave sums.
__global__ __launch_bounds__(64) void gauss_tilted_finish(int nblk, int B, int D, const double *__restrict__ part,
                                                          const double *__restrict__ sn, double alpha,
                                                          double scale, double *__restrict__ scal) {
  const int b = threadIdx.x;
  double lz = b < nblk ? part[2 * b] : 0.0, sdv = b < nblk ? part[2 * b + 1] : 0.0;
  lz = gpx_wave_sum(lz);
  sdv = gpx_wave_sum(sdv);
  if (b != 0) return;
  const double sn2 = exp(2.0 * sn[0]);
  const double two_pi = 6.283185307179586;
  lz += (double)B * D * (0.5 * log(two_pi * sn2 / alpha) - 0.5 * alpha * log(two_pi * sn2));
  scal[0] = lz;
  scal[1] = (sdv * 2.0 * sn2 / alpha + (double)B * D * (1.0 - alpha)) * scale;
}

// SGPSSM.compute_transition_tilted, 2-D branch (aep_models.py:1317-1343).
// Outputs are already scaled; dmall = dmprop - 2 dvprop mprop for the MM adjoint.
// Up to 64 blocks; part[2b], part[2b+1] = block b's (logZ, sum dv) partials.  Bound by the latency of
// an element's log and divisions, as gauss_tilted_kernel (40000 elements 6.7 -> 5.9 us).
__global__ __launch_bounds__(1024) void transition_kernel(int B, int D, const double *__restrict__ mp,
                                                          const double *__restrict__ vp,
                                                          const double *__restrict__ mt,
                                                          const double *__restrict__ vt,
                                                          const double *__restrict__ sn, double alpha,
                                                          double scale, double *__restrict__ dmall,
                                                          double *__restrict__ dvp,
                                                          double *__restrict__ dmt,
                                                          double *__restrict__ dvt,
                                                          double *__restrict__ part) {
  __shared__ double red[16];
  const double sn2 = exp(2.0 * sn[0]);
  const double two_pi = 6.283185307179586;
  double lz = 0.0, sdv = 0.0;
  const long n = (long)B * D;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const double vs = vt[e] + vp[e] + sn2 / alpha;
    const double md = mt[e] - mp[e];
    lz += -0.5 * md * md / vs - 0.5 * log(1.0 + alpha * (vt[e] + vp[e]) / sn2) -
          0.5 * alpha * log(two_pi * sn2);
    const double gv = scale * (-0.5 / vs + 0.5 * md * md / (vs * vs));
    const double gmt = scale * (-md / vs);
    sdv += gv;
    dvt[e] = gv;
    dvp[e] = gv;
    dmt[e] = gmt;
    dmall[e] = -gmt - 2.0 * gv * mp[e];
  }
  lz = gpx_block_sum(lz, red);
  sdv = gpx_block_sum(sdv, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = lz;
    part[2 * blockIdx.x + 1] = sdv;
  }
}

// One wave, lane b holding block b's partials (nblk <= 64), then fixed-order wave sums.
__global__ __launch_bounds__(64) void transition_finish(int nblk, int B, int D, const double *__restrict__ part,
                                                        const double *__restrict__ sn, double alpha,
                                                        double scale, double *__restrict__ scal) {
  const int b = threadIdx.x;
  double lz = b < nblk ? part[2 * b] : 0.0, sdv = b < nblk ? part[2 * b + 1] : 0.0;
  lz = gpx_wave_sum(lz);
  sdv = gpx_wave_sum(sdv);
  if (b != 0) return;
  const double sn2 = exp(2.0 * sn[0]);
  scal[0] = scale * lz;
  scal[1] = sdv * 2.0 * sn2 / alpha + scale * (double)B * D * (1.0 - alpha);
}

// Gauss_Emis.compute_emission_tilted (lik_layers.py:573-627) for Dout <= 8, one thread
// per time step; DT = Dout fixed at compile time, so Vy, its Cholesky factor, the factor's
// inverse and Vy^{-1} live in registers (fully unrolled, lower triangles packed).
// part[blk] collects [logZ, dC (Dout x Din), dR (Dout)] sums over the block's 64 steps
// (unscaled), summed with wave reductions.
constexpr int EM_T = 64;
constexpr int EM_DMAX = 8;
// DI: the row length of C kept in LDS, Din rounded up to 4 or 8 with zeros (0: any Din, its
// loops at run time).  Bound by latency: Nb / 64 waves are less than one per SIMD up to Nb =
// 65,000.  So a step's mx, vx and y are in registers before the algebra, the loops over Din are
// unrolled (their sums and the wave sums interleave), the wave sums land in one lane each and
// are stored together, and dvx reuses dC's product: Nb = 10000, Dout = 8, Din = 4
// 37 -> 19 us (with the finish 47 -> 23).
template <int DT, int DI>
__global__ __launch_bounds__(EM_T) void emission_kernel(int Nb, int Din, const double *__restrict__ C,
                                                        const double *__restrict__ Rp,
                                                        const double *__restrict__ y, int ldy,
                                                        const double *__restrict__ mx, int ldm,
                                                        const double *__restrict__ vx, int ldv,
                                                        double alpha, double scale,
                                                        double *__restrict__ dmx, double *__restrict__ dvx,
                                                        double *__restrict__ part) {
  constexpr int NL = DT * (DT + 1) / 2;
  constexpr int DR = DI ? DI : 1;
  __shared__ double Cs[EM_DMAX * EM_DMAX];
  __shared__ double Rs[EM_DMAX];
  const int tid = threadIdx.x, t = blockIdx.x * EM_T + tid;
  const int ldc = DI ? DI : Din;
  if (DI) {
    if (tid < DT * DI) Cs[tid] = tid % DR < Din ? C[tid / DR * Din + tid % DR] : 0.0;
  } else {
    for (int e = tid; e < DT * Din; e += EM_T) Cs[e] = C[e];
  }
  if (tid < DT) Rs[tid] = exp(2.0 * Rp[tid]);
  const bool ok = t < Nb;
  const int tt = ok ? t : Nb - 1;  // padding steps compute a real step's values, weighted 0
  const double wgt = ok ? 1.0 : 0.0;
  const double *vt = vx + (long)tt * ldv, *mt = mx + (long)tt * ldm;
  double mr[DR], vr[DR], r[DT], u[DT];
  if (DI) {
#pragma unroll
    for (int c = 0; c < DR; ++c) {  // loads at clamped columns, without a branch; zero past Din
      const double m = mt[c < Din ? c : Din - 1], v = vt[c < Din ? c : Din - 1];
      mr[c] = c < Din ? m : 0.0;
      vr[c] = c < Din ? v : 0.0;
    }
  }
#define MT(c) (DI ? mr[DI ? (c) : 0] : mt[c])
#define VT(c) (DI ? vr[DI ? (c) : 0] : vt[c])
#pragma unroll
  for (int a = 0; a < DT; ++a) r[a] = y[(long)tt * ldy + a];
  __syncthreads();
#define LI(a, b) ((a) * ((a) + 1) / 2 + (b))
  // Vy = diag(R/alpha) + C diag(vx) C^T (lower triangle)
  double L[NL];
#pragma unroll
  for (int a = 0; a < DT; ++a)
#pragma unroll
    for (int b = 0; b <= a; ++b) {
      double sum = 0.0;
#pragma unroll
      for (int c = 0; c < ldc; ++c) sum += Cs[a * ldc + c] * VT(c) * Cs[b * ldc + c];
      if (a == b) sum += Rs[a] / alpha;
      L[LI(a, b)] = sum;
    }
  // Cholesky (lower) in place
  double logdetV = 0.0;
#pragma unroll
  for (int k = 0; k < DT; ++k) {
    double sum = L[LI(k, k)];
#pragma unroll
    for (int j = 0; j < k; ++j) sum -= L[LI(k, j)] * L[LI(k, j)];
    const double lkk = sqrt(sum);
    L[LI(k, k)] = lkk;
    logdetV += 2.0 * log(lkk);
#pragma unroll
    for (int i = k + 1; i < DT; ++i) {
      double v = L[LI(i, k)];
#pragma unroll
      for (int j = 0; j < k; ++j) v -= L[LI(i, j)] * L[LI(k, j)];
      L[LI(i, k)] = v / lkk;
    }
  }
  // r = y - C mx;  u = Vy^{-1} r
#pragma unroll
  for (int a = 0; a < DT; ++a)
#pragma unroll
    for (int c = 0; c < ldc; ++c) r[a] -= Cs[a * ldc + c] * MT(c);
#pragma unroll
  for (int a = 0; a < DT; ++a) {  // forward
    double v = r[a];
#pragma unroll
    for (int j = 0; j < a; ++j) v -= L[LI(a, j)] * u[j];
    u[a] = v / L[LI(a, a)];
  }
#pragma unroll
  for (int a = DT - 1; a >= 0; --a) {  // backward
    double v = u[a];
#pragma unroll
    for (int j = a + 1; j < DT; ++j) v -= L[LI(j, a)] * u[j];
    u[a] = v / L[LI(a, a)];
  }
  // Li = L^{-1} (lower), then Vinv = Li^T Li (lower triangle; symmetric)
  double Li[NL];
#pragma unroll
  for (int j = 0; j < DT; ++j)
#pragma unroll
    for (int i = j; i < DT; ++i) {
      double v = (i == j) ? 1.0 : 0.0;
#pragma unroll
      for (int k = j; k < i; ++k) v -= L[LI(i, k)] * Li[LI(k, j)];
      Li[LI(i, j)] = v / L[LI(i, i)];
    }
  double Vi[NL];
#pragma unroll
  for (int a = 0; a < DT; ++a)
#pragma unroll
    for (int b = 0; b <= a; ++b) {
      double v = 0.0;
#pragma unroll
      for (int k = a; k < DT; ++k) v += Li[LI(k, a)] * Li[LI(k, b)];
      Vi[LI(a, b)] = v;
    }
#define VI(a, b) ((a) >= (b) ? Vi[LI(a, b)] : Vi[LI(b, a)])
  double quad = 0.0, sumlogR = 0.0;
#pragma unroll
  for (int a = 0; a < DT; ++a) {
    quad += r[a] * u[a];
    sumlogR += log(Rs[a]);
  }
  // logdet(I + alpha C V C^T / R) = logdet(Vy) + Dout log(alpha) - sum log R
  const double vlog = logdetV + DT * log(alpha) - sumlogR;
  double part0 = -0.5 * quad - 0.5 * vlog - 0.5 * DT * alpha * log(6.283185307179586) - 0.5 * alpha * sumlogR;
  // the block's sums: lane e keeps sum e (and e + 64)
  double keep[2] = {gpx_wave_sum(wgt * part0), 0.0};
  // dSigma = S = -Vinv/2 + u u^T / 2
#define SG(a, b) (-0.5 * VI(a, b) + 0.5 * u[a] * u[b])
#pragma unroll
  for (int a = 0; a < DT; ++a) {
    const double dr = gpx_wave_sum(wgt * SG(a, a));
    const int e = 1 + DT * Din + a;
    keep[0] = tid == e ? dr : keep[0];
    keep[1] = tid + EM_T == e ? dr : keep[1];
  }
#pragma unroll
  for (int c = 0; c < ldc; ++c) {
    double gm = 0.0, gv = 0.0;
#pragma unroll
    for (int a = 0; a < DT; ++a) {
      double v = 0.0;  // (S C)[a][c]
#pragma unroll
      for (int b = 0; b < DT; ++b) v += SG(a, b) * Cs[b * ldc + c];
      gm += u[a] * Cs[a * ldc + c];
      gv += v * Cs[a * ldc + c];
      const double dc = gpx_wave_sum(wgt * (u[a] * MT(c) + 2.0 * v * VT(c)));
      const int e = 1 + a * Din + c;
      keep[0] = tid == e && c < Din ? dc : keep[0];
      keep[1] = tid + EM_T == e && c < Din ? dc : keep[1];
    }
    if (ok && c < Din) {
      dmx[(long)t * Din + c] = gm * scale;
      dvx[(long)t * Din + c] = gv * scale;
    }
  }
  const int W = DT * Din + DT + 1;
  double *pb = part + (long)blockIdx.x * W;
  if (tid < W) pb[tid] = keep[0];
  if (tid + EM_T < W) pb[tid + EM_T] = keep[1];
#undef SG
#undef MT
#undef VT
#undef VI
#undef LI
}

// logZ, dC, dR from the block partials (the dR chain of lik_layers.py:610-613), a wave per
// sum: lane l adds blocks l, l + 64, ... in order, then the wave's lanes.
__global__ __launch_bounds__(64) void emission_final(int nblk, int Nb, int Dout, int Din,
                                                     const double *__restrict__ part,
                                                     const double *__restrict__ Rp, double alpha, double scale,
                                                     double *__restrict__ dC, double *__restrict__ dR,
                                                     double *__restrict__ scal) {
  const int W = Dout * Din + Dout + 1, i = blockIdx.x;
  double s = 0.0;
#pragma unroll 4
  for (int b = threadIdx.x; b < nblk; b += 64) s += part[(long)b * W + i];
  s = gpx_wave_sum(s);
  if (threadIdx.x != 0) return;
  if (i == 0) {
    scal[0] = s * scale;
  } else if (i <= Dout * Din) {
    dC[i - 1] = s * scale;
  } else {
    const int a = i - 1 - Dout * Din;
    const double R = exp(2.0 * Rp[a]);
    const double g = s / alpha + 0.5 * Nb * (1.0 - alpha) / R;
    dR[a] = g * 2.0 * R * scale;
  }
}

// out[n][m] = alpha sum_d w[n, d] T[d][n][m] + beta out[n][m]   (aep_models.py:455)
__global__ void wsum_kernel(int N, int D, int M, double alpha, const double *__restrict__ w,
                            const double *__restrict__ T, double beta, double *__restrict__ out) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const long NM = (long)N * M;
  if (e >= NM) return;
  const int n = (int)(e / M);
  double s = 0.0;
#pragma unroll 8
  for (int d = 0; d < D; ++d) s += w[(long)n * D + d] * T[(long)d * NM + e];
  out[e] = (beta == 0.0) ? alpha * s : alpha * s + beta * out[e];
}

// out = dm - 2 dv m   (aep_models.py:235)
__global__ void dmall_kernel(long n, const double *__restrict__ dm, const double *__restrict__ dv,
                             const double *__restrict__ m, double *__restrict__ out) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e < n) out[e] = dm[e] - 2.0 * dv[e] * m[e];
}

// dls = dell * exp(ls) + 2 gls;  dsf = 2 exp(2 sf) (dsf2 + sumdv) + 2 gsf
// (aep_models.py:244-247, 296-298, 456-460, 502-504)
__global__ void hyper_kernel(int Q, const double *__restrict__ ls, const double *__restrict__ sf,
                             const double *__restrict__ dell, const double *__restrict__ gls,
                             const double *__restrict__ dsf2, const double *__restrict__ sumdv,
                             const double *__restrict__ gsf, double *__restrict__ dls,
                             double *__restrict__ dsf) {
  const int q = threadIdx.x;
  if (q < Q) dls[q] = dell[q] * exp(ls[q]) + 2.0 * gls[q];
  if (q == 0) dsf[0] = 2.0 * exp(2.0 * sf[0]) * (dsf2[0] + sumdv[0]) + 2.0 * gsf[0];
}

// phi = (D/2) ldK + sp/2 sum_d (sp_sign ldP_d + dotP_d) + sc/2 sum_d (sc_sign ldC_d + dotC_d)
// (aep_models.py:62-114)
__global__ void phi_kernel(int D, const double *__restrict__ ldK, const double *__restrict__ ldP,
                           double sgnP, const double *__restrict__ dotP, const double *__restrict__ ldC,
                           double sgnC, const double *__restrict__ dotC, double sp, double sc,
                           double *__restrict__ out) {
  if (threadIdx.x != 0) return;
  double p = 0.0, c = 0.0;
  for (int d = 0; d < D; ++d) {
    p += sgnP * ldP[d] + dotP[d];
    c += sgnC * ldC[d] + dotC[d];
  }
  out[0] = D * 0.5 * ldK[0] + sp * 0.5 * p + sc * 0.5 * c;
}

// Natural-parameter phi with the quadratic terms taken from theta2: Sigma^-1 mu = theta2
// and Sigma-hat^-1 mu-hat = beta theta2, so mu^T Sigma^-1 mu = mu . theta2 and
// mu-hat^T Sigma-hat^-1 mu-hat = beta mu-hat . theta2.  One workgroup; the partial sums
// and their reduction run in a fixed order.
__global__ __launch_bounds__(256) void phi_nat_kernel(int D, int M, const double *__restrict__ ldK,
                                                      const double *__restrict__ ldP,
                                                      const double *__restrict__ ldC,
                                                      const double *__restrict__ mu,
                                                      const double *__restrict__ muhat,
                                                      const double *__restrict__ th2, double beta,
                                                      double sp, double sc, double *__restrict__ out) {
  __shared__ double red[16];
  double p = 0.0, c = 0.0;
  const long n = (long)D * M;
  for (long e = threadIdx.x; e < n; e += 256) {
    p = fma(mu[e], th2[e], p);
    c = fma(muhat[e], th2[e], c);
  }
  p = gpx_block_sum(p, red);
  c = gpx_block_sum(c, red);
  if (threadIdx.x == 0) {
    double lp = 0.0, lc = 0.0;
    for (int d = 0; d < D; ++d) {
      lp -= ldP[d];
      lc -= ldC[d];
    }
    out[0] = D * 0.5 * ldK[0] + sp * 0.5 * (lp + p) + sc * 0.5 * (lc + beta * c);
  }
}

// my = C mf, vy_d = sum_c C_dc^2 vf_c + R_d (diagonal of lik_layers.py:558-571)
__global__ void emission_predict_kernel(int Nb, int Dout, int Din, const double *__restrict__ C,
                                        const double *__restrict__ Rp, const double *__restrict__ mf,
                                        const double *__restrict__ vf, double *__restrict__ my,
                                        double *__restrict__ vy) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= (long)Nb * Dout) return;
  const int n = (int)(e / Dout), d = (int)(e % Dout);
  double m = 0.0, v = exp(2.0 * Rp[d]);
  for (int c = 0; c < Din; ++c) {
    const double cc = C[d * Din + c];
    m += cc * mf[(long)n * Din + c];
    v += cc * cc * vf[(long)n * Din + c];
  }
  my[e] = m;
  vy[e] = v;
}

// Kuu of several layers of one M in one launch: K[l] = sf2_l exp(-r2 / 2) + jitter I over
// the layer's inducing inputs z_l (M x Q_l), the arithmetic of se_kernel with x = z.
constexpr int kKuuLayers = 16;
struct KuuLayers {
  const double *z[kKuuLayers], *ls[kKuuLayers], *sf[kKuuLayers];
  int Q[kKuuLayers];
};
__global__ __launch_bounds__(256) void kuu_batched_kernel(int nl, KuuLayers L, int M, double jitter,
                                                          double *__restrict__ K) {
  __shared__ double il[16], s2;
  const long MM = (long)M * M;
  const int l = blockIdx.y, Q = L.Q[l];
  const double *z = L.z[l], *ls = L.ls[l];
  if (threadIdx.x < 16) il[threadIdx.x] = (int)threadIdx.x < Q ? exp(-2.0 * ls[threadIdx.x]) : 0.0;
  if (threadIdx.x == 255) s2 = exp(2.0 * L.sf[l][0]);
  __syncthreads();
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= MM) return;
  const int n = (int)(e / M), m = (int)(e % M);
  double r2 = 0.0;
  for (int q = 0; q < Q; ++q) {
    const double d = z[n * Q + q] - z[m * Q + q];
    if (Q <= 16)
      r2 = fma(d * il[q], d, r2);  // the operations of se_kernel
    else
      r2 += d * d / exp(2.0 * ls[q]);  // those of se_any_kernel
  }
  double k = s2 * exp(-0.5 * r2);
  if (n == m) k += jitter;
  K[l * MM + e] = k;
}

// Posterior and cavity precisions of several layers of one M from X = R^T R (the
// layers' output dims stacked) and their Kuu^-1 (stacked): layer l with D_l outputs at
// rows x_l of X writes prec[2 x_l + d] = X[x_l + d] + Ki[l] and prec[2 x_l + D_l + d] =
// beta X[x_l + d] + Ki[l].  One thread per element of X.
constexpr int kPrecLayers = 16;
struct PrecLayers {
  int D[kPrecLayers];
};
__global__ __launch_bounds__(256) void prec_form_kernel(int nl, PrecLayers L, int M, const double *__restrict__ X,
                                                        const double *__restrict__ Ki, double beta,
                                                        double *__restrict__ prec) {
  const long MM = (long)M * M;
  const long e = blockIdx.x * 256L + threadIdx.x;
  int row = (int)(e / MM), l = 0, x0 = 0;
  while (l < nl && row >= x0 + L.D[l]) x0 += L.D[l++];
  if (l >= nl) return;  // past the last layer's rows
  const long m = e - (long)row * MM;
  const double x = X[e], k = Ki[l * MM + m];
  const int d = row - x0;
  prec[(2L * x0 + d) * MM + m] = x + k;
  prec[(2L * x0 + L.D[l] + d) * MM + m] = beta * x + k;
}

}  // namespace

extern "C" {

// K[n,m] = SE(x_n, z_m) (+ jitter on n == m); x is N rows with leading dim ldx.
int gpx_se_kernel(int N, int M, int Q, const double *x, int ldx, const double *z, const double *ls,
                  const double *sf, double jitter, double *K, void *stream) {
  if (N < 0 || M < 0 || Q < 1 || ldx < Q) return GPX_EINVAL;
  if (N == 0 || M == 0) return GPX_OK;
  if (!x || !z || !ls || !sf || !K) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (Q > 16 || M > 64 * 65535) {
    hipLaunchKernelGGL(se_any_kernel, dim3(gpx_cdiv((long)N * M, 256)), dim3(256), 0, st, N, M, Q, x, ldx, z, ls, sf,
                       jitter, K);
  } else {
    const int cb = M <= 16 ? 16 : (M <= 32 ? 32 : 64), step = 256 / cb;
    const bool few = (long)gpx_cdiv(N, 4 * step) * gpx_cdiv(M, cb) <= (Q <= 4 ? 256 : (Q <= 8 ? 192 : 96));
    const dim3 grid(gpx_cdiv(N, (few ? 1 : 4) * step), gpx_cdiv(M, cb));
#define GPX_SE2(QV, CB)                                                                                               \
  do {                                                                                                                \
    if (few) hipLaunchKernelGGL((se_kernel<QV, 1, CB>), grid, dim3(256), 0, st, N, M, Q, x, ldx, z, ls, sf, jitter, K); \
    else hipLaunchKernelGGL((se_kernel<QV, 4, CB>), grid, dim3(256), 0, st, N, M, Q, x, ldx, z, ls, sf, jitter, K);     \
  } while (0)
#define GPX_SE(QV) if (cb == 16) GPX_SE2(QV, 16); else if (cb == 32) GPX_SE2(QV, 32); else GPX_SE2(QV, 64);
    if (Q <= 4) { GPX_SE(4) }
    else if (Q <= 8) { GPX_SE(8) }
    else { GPX_SE(16) }
#undef GPX_SE
#undef GPX_SE2
  }
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// Columns of the adjoint's thread layout, and its number of blocks: eight rows a thread or more, four
// where that makes at most 60 blocks (whole adjoint, us, four : eight: N = 197, M = 64, Q = 15 11.9 : 13.4,
// 953, 22, 13 (60) 11.5 : 12.5, 1000, 50, 2 (63) 9.6 : 9.2, 2000, 200, 16 31 : 27), at most two blocks per CU (their
// partials are read again by pass 2).
static int kfu_cols(int M) { return M <= 64 ? 64 : (M <= 128 ? 128 : 256); }
static int kfu_blocks(int N, int M) {
  const int groups = 256 / kfu_cols(M), four = (int)std::min<long>(512, gpx_cdiv(N, 4L * groups));
  return four <= 60 ? four : (int)std::min<long>(512, gpx_cdiv(N, 8L * groups));
}

long gpx_kfu_bwd_workspace(int N, int M, int Q) { return ((long)kfu_blocks(N, M) + 1) * M * (2 * Q + 1); }

static int kfu_bwd_launch(int N, int M, int Q, const double *dK, const KfuReg *reg, const double *K, const double *x,
                          const double *z, const double *ls, const double *sf, double *dsf2, double *dell, double *dZ,
                          double *dx, double *work, hipStream_t st) {
  const int nblk = kfu_blocks(N, M), MP = kfu_cols(M), W = 2 * Q + 1, rows = reg ? W + 1 : W;
  double *red = work + (long)nblk * M * rows;
#define GPX_KFU(QV)                                                                                           \
  if (reg)                                                                                                    \
    hipLaunchKernelGGL((kfu_bwd_partial<QV, true>), dim3(nblk), dim3(256), 0, st, N, M, Q, MP, dK, *reg, K, x, z, work); \
  else                                                                                                        \
    hipLaunchKernelGGL((kfu_bwd_partial<QV, false>), dim3(nblk), dim3(256), 0, st, N, M, Q, MP, dK, KfuReg{}, K, x, z, \
                       work);
  if (Q <= 4) { GPX_KFU(4) }
  else if (Q <= 8) { GPX_KFU(8) }
  else if (Q <= 12) { GPX_KFU(12) }
  else { GPX_KFU(16) }
#undef GPX_KFU
  GPX_CHECK_LAUNCH();
  const int sums = (int)gpx_cdiv(M, 64) * rows;
#define GPX_KFU_FINAL(KR)                                                                                         \
  hipLaunchKernelGGL(kfu_bwd_final<KR>, dim3(sums + (KR ? gpx_cdiv(N, 16) : 0)), dim3(1024),                          \
                     KR ? M * (Q | 1) * sizeof(double) : 0, st, nblk, M, rows, sums, (const double *)work, red, N, Q, \
                     dK, K, x, z, ls, dx)
  if (!dx) GPX_KFU_FINAL(0);
  else if (Q <= 4) GPX_KFU_FINAL(1);
  else if (Q <= 8) GPX_KFU_FINAL(2);
  else if (Q <= 12) GPX_KFU_FINAL(3);
  else GPX_KFU_FINAL(4);
#undef GPX_KFU_FINAL
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(kfu_bwd_scalars, dim3(Q + 1), dim3(64), 0, st, M, Q, (const double *)red,
                     reg ? (const double *)red + (long)W * M : nullptr, z, ls, sf, dsf2, dell, dZ);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// Adjoint of K(x, Z): dsf2 (w.r.t. sf2), dell (w.r.t. ell), dZ (M x Q), dx (N x Q, optional).
int gpx_kfu_bwd(int N, int M, int Q, const double *dK, const double *K, const double *x,
                const double *z, const double *ls, const double *sf, double *dsf2, double *dell,
                double *dZ, double *dx, double *work, void *stream) {
  if (N < 1 || M < 1 || M > 256 || Q < 1 || Q > 16) return GPX_EINVAL;
  if (!dK || !K || !x || !z || !ls || !sf || !dsf2 || !dell || !dZ || !work) return GPX_EINVAL;
  return kfu_bwd_launch(N, M, Q, dK, nullptr, K, x, z, ls, sf, dsf2, dell, dZ, dx, work, (hipStream_t)stream);
}

long gpx_kfu_bwd_reg_workspace(int N, int M, int Q) { return ((long)kfu_blocks(N, M) + 1) * M * (2 * Q + 2); }

int gpx_kfu_bwd_reg(int N, int D, int M, int Q, const double *dm, const double *dv, const double *A, const double *T,
                    const double *K, const double *x, const double *z, const double *ls, const double *sf, double *dsf2,
                    double *dell, double *dZ, double *work, void *stream) {
  if (N < 1 || D < 1 || M < 1 || M > 256 || Q < 1 || Q > 16) return GPX_EINVAL;
  if (!dm || !dv || !A || !T || !K || !x || !z || !ls || !sf || !dsf2 || !dell || !dZ || !work) return GPX_EINVAL;
  const KfuReg reg{D, dm, dv, A, T};
  return kfu_bwd_launch(N, M, Q, nullptr, &reg, K, x, z, ls, sf, dsf2, dell, dZ, nullptr, work, (hipStream_t)stream);
}

long gpx_dtrace_workspace(int M, int Q) { return (long)M * (Q + 1); }

static int launch_dtrace(int M, int Q, const double *Mm, const double *z, const double *ls, const double *sf,
                         const double *dz0, double *gz, double *work, hipStream_t st) {
  switch (Q) {
#define GPX_DT(QV)                                                                                               \
  case QV:                                                                                                       \
    hipLaunchKernelGGL((dtrace_kernel<QV>), dim3(gpx_cdiv(M, 4)), dim3(256), 0, st, M, Mm, z, ls, sf, dz0, gz, work); \
    break;
    GPX_DT(1) GPX_DT(2) GPX_DT(3) GPX_DT(4) GPX_DT(5) GPX_DT(6) GPX_DT(7) GPX_DT(8)
    GPX_DT(9) GPX_DT(10) GPX_DT(11) GPX_DT(12) GPX_DT(13) GPX_DT(14) GPX_DT(15) GPX_DT(16)
#undef GPX_DT
  }
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// d tr(Mm Kzz) / d(lsf, lls, z) for Kzz = SE(z, z): gsf (1), gls (Q), gz (M x Q).
int gpx_dtrace_kzz(int M, int Q, const double *Mm, const double *z, const double *ls,
                   const double *sf, double *gsf, double *gls, double *gz, double *work,
                   void *stream) {
  if (M < 1 || M > 256 || Q < 1 || Q > 16 || !Mm || !z || !ls || !sf || !gsf || !gls || !gz || !work)
    return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const int rc = launch_dtrace(M, Q, Mm, z, ls, sf, nullptr, gz, work, st);
  if (rc != GPX_OK) return rc;
  hipLaunchKernelGGL(dtrace_final, dim3(Q + 1), dim3(64), 0, st, M, Q, (const double *)work, gsf, gls);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_kuu_tail(int M, int Q, const double *Mm, const double *z, const double *ls, const double *sf,
                 const double *dell, const double *dsf2, const double *sumdv, const double *dz0, double *dls,
                 double *dsf, double *dZ, double *work, void *stream) {
  if (M < 1 || M > 256 || Q < 1 || Q > 16 || !Mm || !z || !ls || !sf || !dell || !dsf2 || !dz0 || !dls ||
      !dsf || !dZ || !work)
    return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const int rc = launch_dtrace(M, Q, Mm, z, ls, sf, dz0, dZ, work, st);
  if (rc != GPX_OK) return rc;
  hipLaunchKernelGGL(kuu_tail_kernel, dim3(Q + 1), dim3(64), 0, st, M, Q, (const double *)work, ls, sf, dell, dsf2,
                     sumdv, dls, dsf);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_moments(int batch, int D, int M, const double *S, const double *theta, double s0, double s1, double *mu,
                double *P, void *stream) {
  if (batch < 0 || D < 1 || M < 1 || M > 256) return GPX_EINVAL;
  if (batch == 0) return GPX_OK;
  if (!S || !theta || !mu || !P) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (M <= 64) {
    hipLaunchKernelGGL(moments_kernel, dim3(batch), dim3(1024), 0, st, D, M, S, theta, s0, s1, mu, P);
    GPX_CHECK_LAUNCH();
    return GPX_OK;
  }
  hipLaunchKernelGGL(mean_kernel, dim3(batch, gpx_cdiv(M, 4)), dim3(256), 0, st, D, M, S, theta, s0, s1, mu);
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(second_kernel, dim3(batch, gpx_cdiv(M * M, 256)), dim3(256), 0, st, M, S, (const double *)mu, P);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// out[j] = alpha * sum_i P[i, j] + beta * out[j]
int gpx_colsum(int rows, int cols, const double *P, double alpha, double beta, double *out, void *stream) {
  if (rows < 0 || cols < 0 || !P || !out) return GPX_EINVAL;
  if (cols == 0) return GPX_OK;
  if (rows >= 512 && cols <= 1024) {
    hipLaunchKernelGGL(colsum_tall_kernel, dim3(cols), dim3(256), 0, (hipStream_t)stream, rows, cols, P, alpha,
                       beta, out);
    GPX_CHECK_LAUNCH();
    return GPX_OK;
  }
  hipLaunchKernelGGL(colsum_kernel, dim3(gpx_cdiv(cols, 256)), dim3(256), 0, (hipStream_t)stream, rows, cols,
                     P, alpha, beta, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// Chunks of the two-stage column sum and its workspace (doubles).
static int colsum_chunks(int rows) {
  int c = (rows + 2047) / 2048;
  return c > 256 ? 256 : c;
}

long gpx_colsum_workspace(int rows, int cols) {
  if (rows < 0 || cols < 0) return -1;
  return (long)colsum_chunks(rows) * cols;
}

// out[j] = alpha sum_i P[i, j] + beta out[j] for tall P: chunked partial sums into
// `work`, then their fixed-order sum; the same result for the same input and shape.
int gpx_colsum_tall(int rows, int cols, const double *P, double alpha, double beta, double *out, double *work,
                    void *stream) {
  if (rows < 0 || cols < 0 || cols > 65535 || !P || !out || !work) return GPX_EINVAL;
  if (cols == 0) return GPX_OK;
  const int nc = colsum_chunks(rows > 0 ? rows : 1);
  const int chunk = (rows + nc - 1) / nc;
  hipLaunchKernelGGL(colsum_chunk_kernel, dim3(cols, nc), dim3(256), 0, (hipStream_t)stream, rows, cols, chunk, P,
                     work);
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(colsum_kernel, dim3(gpx_cdiv(cols, 256)), dim3(256), 0, (hipStream_t)stream, nc, cols,
                     (const double *)work, alpha, beta, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_eta_to_R(int D, int M, const double *eta, double *R, void *stream) {
  if (D < 0 || M < 1 || !eta || !R) return GPX_EINVAL;
  long n = (long)D * M * M;
  if (n == 0) return GPX_OK;
  hipLaunchKernelGGL(eta_to_R_kernel, dim3(gpx_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, D, M, eta, R);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_kuu_batched(int nl, int M, const double *const *z, const int *Q, const double *const *ls,
                    const double *const *sf, double jitter, double *K, void *stream) {
  if (nl < 1 || nl > kKuuLayers || M < 1 || !z || !Q || !ls || !sf || !K) return GPX_EINVAL;
  KuuLayers L = {};
  for (int l = 0; l < nl; ++l) {
    if (!z[l] || !ls[l] || !sf[l] || Q[l] < 1) return GPX_EINVAL;
    L.z[l] = z[l];
    L.ls[l] = ls[l];
    L.sf[l] = sf[l];
    L.Q[l] = Q[l];
  }
  hipLaunchKernelGGL(kuu_batched_kernel, dim3(gpx_cdiv((long)M * M, 256), nl), dim3(256), 0, (hipStream_t)stream, nl,
                     L, M, jitter, K);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_prec_form(int nl, const int *D, int M, const double *X, const double *Ki, double beta, double *prec,
                  void *stream) {
  if (nl < 1 || nl > kPrecLayers || !D || M < 1 || !X || !Ki || !prec) return GPX_EINVAL;
  PrecLayers L = {};
  long rows = 0;
  for (int l = 0; l < nl; ++l) {
    if (D[l] < 1) return GPX_EINVAL;
    L.D[l] = D[l];
    rows += D[l];
  }
  hipLaunchKernelGGL(prec_form_kernel, dim3(gpx_cdiv(rows * M * M, 256)), dim3(256), 0, (hipStream_t)stream, nl, L,
                     M, X, Ki, beta, prec);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_pack_dR(int D, int M, const double *R, const double *G, double *out, void *stream) {
  if (D < 0 || M < 1 || !R || !G || !out) return GPX_EINVAL;
  long n = (long)D * M * (M + 1) / 2;
  if (n == 0) return GPX_OK;
  if (D > 65535) return GPX_EINVAL;
  const int MT = (M + 15) / 16;
  hipLaunchKernelGGL(pack_dR_kernel, dim3(MT * (MT + 1) / 2, D), dim3(256), 0, (hipStream_t)stream, D, M, R, G,
                     out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// out[i] = a x[i % nx] + b y[i % ny] + c w[i % nw]  (y, w optional); out may alias inputs.
int gpx_lincomb(long n, double a, const double *x, long nx, double b, const double *y, long ny,
                double c, const double *w, long nw, double *out, void *stream) {
  if (n < 0 || !x || nx < 1 || !out || (y && ny < 1) || (w && nw < 1)) return GPX_EINVAL;
  if (n == 0) return GPX_OK;
  unsigned g = gpx_cdiv(n, 256);
  if (g > 8192) g = 8192;
  hipLaunchKernelGGL(lincomb_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, n, a, x, nx, b, y, ny, c, w,
                     nw, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// out[b] = a (X[b] + X[b]^T); out must not alias X.
int gpx_sym(int batch, int M, double a, const double *X, double *out, void *stream) {
  if (batch < 0 || M < 0 || !X || !out || X == out) return GPX_EINVAL;
  long n = (long)batch * M * M;
  if (n == 0) return GPX_OK;
  hipLaunchKernelGGL(sym_kernel, dim3(gpx_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, batch, M, a, X, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_det_var(int N, int D, int M, const double *T, const double *kfu, const double *sf, double *v,
                void *stream) {
  if (N < 0 || D < 0 || M < 1 || !T || !kfu || !sf || !v) return GPX_EINVAL;
  long n = (long)N * D;
  if (n == 0) return GPX_OK;
  hipLaunchKernelGGL(det_var_kernel, dim3(gpx_cdiv(n, 4)), dim3(256), 0, (hipStream_t)stream, N, D, M, T, kfu,
                     sf, v);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_mm_var(long n, const double *m, const double *Bp, const double *sf, double *v, void *stream) {
  if (n < 0 || !m || !Bp || !sf || !v) return GPX_EINVAL;
  if (n == 0) return GPX_OK;
  hipLaunchKernelGGL(mm_var_kernel, dim3(gpx_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, n, m, Bp, sf, v);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_batched_dot(int batch, int n, const double *x, const double *y, double *out, void *stream) {
  if (batch < 0 || n < 0 || !x || !y || !out) return GPX_EINVAL;
  if (batch == 0) return GPX_OK;
  hipLaunchKernelGGL(batched_dot_kernel, dim3(batch), dim3(256), 0, (hipStream_t)stream, batch, n, x, y, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// scal needs 2 + 2 * 64 doubles: [logZ, dsn] followed by per-block partials.
int gpx_gauss_tilted(int B, int D, const double *m, const double *v, const double *y, const double *sn,
                     double alpha, double scale, double *dm, double *dv, double *dmall, double *scal,
                     void *stream) {
  if (B < 1 || D < 1 || !(alpha > 0) || !m || !v || !y || !sn || !dm || !dv || !scal) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  long n = (long)B * D;
  const int threads = gpx_even_threads(n), nblk = (int)std::min<long>(64, gpx_cdiv(n, threads));
  hipLaunchKernelGGL(gauss_tilted_kernel, dim3(nblk), dim3(threads), 0, st, B, D, m, v, y, sn, alpha, scale, dm, dv,
                     dmall, scal + 2);
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(gauss_tilted_finish, dim3(1), dim3(64), 0, st, nblk, B, D, (const double *)(scal + 2), sn,
                     alpha, scale, scal);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_transition_tilted(int B, int D, const double *mp, const double *vp, const double *mt,
                          const double *vt, const double *sn, double alpha, double scale,
                          double *dmall, double *dvp, double *dmt, double *dvt, double *scal,
                          void *stream) {
  if (B < 1 || D < 1 || !(alpha > 0) || !mp || !vp || !mt || !vt || !sn || !dmall || !dvp || !dmt ||
      !dvt || !scal)
    return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  long n = (long)B * D;
  const int nt = gpx_even_threads(n);
  int nblk = (int)gpx_cdiv(n, nt);
  if (nblk > 64) nblk = 64;
  hipLaunchKernelGGL(transition_kernel, dim3(nblk), dim3(nt), 0, st, B, D, mp, vp, mt, vt, sn, alpha, scale, dmall,
                     dvp, dmt, dvt, scal + 2);
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(transition_finish, dim3(1), dim3(64), 0, st, nblk, B, D, (const double *)(scal + 2), sn,
                     alpha, scale, scal);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

long gpx_emission_workspace(int Nb, int Dout, int Din) {
  return (long)gpx_cdiv(Nb, EM_T) * (Dout * Din + Dout + 1);
}

int gpx_emission_tilted(int Nb, int Dout, int Din, const double *C, const double *Rp, const double *y,
                        int ldy, const double *mx, int ldm, const double *vx, int ldv, double alpha,
                        double scale, double *dmx, double *dvx, double *dC, double *dR, double *scal,
                        double *work, void *stream) {
  if (Nb < 1 || Dout < 1 || Dout > EM_DMAX || Din < 1 || !(alpha > 0)) return GPX_EINVAL;
  if (!C || !Rp || !y || !mx || !vx || !dmx || !dvx || !dC || !dR || !scal || !work) return GPX_EINVAL;
  if (Dout * Din > EM_DMAX * EM_DMAX || Dout * Din + Dout + 2 > EM_DMAX * EM_DMAX + EM_DMAX + 2)
    return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const unsigned nblk = gpx_cdiv(Nb, EM_T);
#define GPX_EMIS1(DTV, DIV)                                                                                        \
  hipLaunchKernelGGL((emission_kernel<DTV, DIV>), dim3(nblk), dim3(EM_T), 0, st, Nb, Din, C, Rp, y, ldy, mx, ldm, \
                     vx, ldv, alpha, scale, dmx, dvx, work)
#define GPX_EMIS(DTV)          \
  do {                         \
    if (Din <= 4)              \
      GPX_EMIS1(DTV, 4);       \
    else if (Din <= 8)         \
      GPX_EMIS1(DTV, 8);       \
    else                       \
      GPX_EMIS1(DTV, 0);       \
  } while (0)
  switch (Dout) {
    case 1: GPX_EMIS(1); break;
    case 2: GPX_EMIS(2); break;
    case 3: GPX_EMIS(3); break;
    case 4: GPX_EMIS(4); break;
    case 5: GPX_EMIS(5); break;
    case 6: GPX_EMIS(6); break;
    case 7: GPX_EMIS(7); break;
    default:  // Dout Din <= 64
      if (Din <= 4)
        GPX_EMIS1(8, 4);
      else
        GPX_EMIS1(8, 8);
  }
#undef GPX_EMIS
#undef GPX_EMIS1
  GPX_CHECK_LAUNCH();
  hipLaunchKernelGGL(emission_final, dim3(Dout * Din + Dout + 1), dim3(64), 0, st, (int)nblk, Nb, Dout, Din, (const double *)work,
                     Rp, alpha, scale, dC, dR, scal);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_wsum(int N, int D, int M, double alpha, const double *w, const double *T, double beta,
             double *out, void *stream) {
  if (N < 0 || D < 0 || M < 0 || !w || !T || !out) return GPX_EINVAL;
  long n = (long)N * M;
  if (n == 0) return GPX_OK;
  hipLaunchKernelGGL(wsum_kernel, dim3(gpx_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, N, D, M, alpha, w, T,
                     beta, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_dmall(long n, const double *dm, const double *dv, const double *m, double *out, void *stream) {
  if (n < 0 || !dm || !dv || !m || !out) return GPX_EINVAL;
  if (n == 0) return GPX_OK;
  hipLaunchKernelGGL(dmall_kernel, dim3(gpx_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, n, dm, dv, m, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_hyper_grads(int Q, const double *ls, const double *sf, const double *dell, const double *gls,
                    const double *dsf2, const double *sumdv, const double *gsf, double *dls, double *dsf,
                    void *stream) {
  if (Q < 1 || Q > 1024 || !ls || !sf || !dell || !gls || !dsf2 || !sumdv || !gsf || !dls || !dsf)
    return GPX_EINVAL;
  hipLaunchKernelGGL(hyper_kernel, dim3(1), dim3(Q < 64 ? 64 : ((Q + 63) / 64) * 64), 0, (hipStream_t)stream, Q,
                     ls, sf, dell, gls, dsf2, sumdv, gsf, dls, dsf);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_phi(int D, const double *ldK, const double *ldP, double sgnP, const double *dotP,
            const double *ldC, double sgnC, const double *dotC, double sp, double sc, double *out,
            void *stream) {
  if (D < 1 || !ldK || !ldP || !dotP || !ldC || !dotC || !out) return GPX_EINVAL;
  hipLaunchKernelGGL(phi_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, D, ldK, ldP, sgnP, dotP, ldC, sgnC,
                     dotC, sp, sc, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_phi_nat(int D, int M, const double *ldK, const double *ldP, const double *ldC, const double *mu,
                const double *muhat, const double *theta2, double beta, double sp, double sc, double *out,
                void *stream) {
  if (D < 1 || M < 1 || !ldK || !ldP || !ldC || !mu || !muhat || !theta2 || !out) return GPX_EINVAL;
  hipLaunchKernelGGL(phi_nat_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, D, M, ldK, ldP, ldC, mu,
                     muhat, theta2, beta, sp, sc, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

int gpx_emission_predict(int Nb, int Dout, int Din, const double *C, const double *Rp, const double *mf,
                         const double *vf, double *my, double *vy, void *stream) {
  if (Nb < 0 || Dout < 1 || Din < 1 || !C || !Rp || !mf || !vf || !my || !vy) return GPX_EINVAL;
  if (Nb == 0) return GPX_OK;
  hipLaunchKernelGGL(emission_predict_kernel, dim3(gpx_cdiv((long)Nb * Dout, 256)), dim3(256), 0,
                     (hipStream_t)stream, Nb, Dout, Din, C, Rp, mf, vf, my, vy);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

}  // extern "C"
