// Batched, strided FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4f64).
//
// Row-major C[b] = alpha * op(A[b]) * op(B[b]) + beta * C[b].  It carries every dense
// contraction of the layer algebra that the reference writes as np.dot / np.einsum
// over D x M x M stacks (aep_models.py:156, 197, 239-258, 453-493, 525-546;
// base_models.py:470-488, 497), including the N x M^2 projections of psi2.
// Split-K partial slabs (one per z-slice of the grid) are summed by a deterministic
// second pass, so results do not depend on scheduling.
#include "gpx_frag.h"
#include "../../include/gpx.h"

namespace {

// Output epilogue: C = v + beta C + gamma E (beta == 0 never reads C; E may be NULL; an
// E stride of 0 broadcasts one matrix over the batch).  With a tail (EXT kernels): the outer
// products delta sum_t U_t V_t^T are added, to C or, if there is a C2, to C2 = a2 (C + outer) + E2.
struct GemmEpi {
  double beta, gamma;
  const double *E;
  int ldE;
  long sE;
  int ext;      // whether `t` counts
  int um, vn;   // its rows: m, n
  GpxGemmTail t;
};

// Terms t0, t0 + step, ... of the tail's sum_t U_t[i] V_t[j].
__device__ __forceinline__ double epi_outer(const GemmEpi &ep, int b, int i, int j, int t0, int step) {
  const double *u = ep.t.U + b * ep.t.sU + i, *w = ep.t.V + b * ep.t.sV + j;
  double s = 0.0;
#pragma unroll 4
  for (int t = t0; t < ep.t.terms; t += step) s = fma(u[(long)t * ep.um], w[(long)t * ep.vn], s);
  return s;
}

// `outer`: epi_outer over all terms (formed here unless the caller has it).
template <bool EXT, bool HAVE = false>
__device__ __forceinline__ void epi_store(double *c, double v, const GemmEpi &ep, int b, int i, int j,
                                          double outer = 0.0) {
  double r = v;
  if (ep.beta != 0.0) r += ep.beta * *c;
  if (ep.E) r += ep.gamma * ep.E[b * ep.sE + (long)i * ep.ldE + j];
  if constexpr (EXT) {
    if (ep.ext) {
      const double s = r + ep.t.delta * (HAVE ? outer : epi_outer(ep, b, i, j, 0, 1));
      if (ep.t.C2) {
        const long e = (long)i * ep.vn + j;
        ep.t.C2[b * ep.t.sC2 + e] = ep.t.E2 ? ep.t.a2 * s + ep.t.E2[b * ep.t.sE2 + e] : ep.t.a2 * s;
      } else {
        r = s;
      }
    }
  }
  *c = r;
}

// Sum of the split-K partials part[q][b][i][j] (q < splits) and the epilogue.  A workgroup
// takes 32 consecutive outputs; its 8 groups of 32 threads each sum the splits q = g,
// g + 8, ... of them (coalesced rows, loads in flight together), and the 8 group sums are
// added in group order, so every output's order of summation is fixed.  splits = 0 (k = 0)
// stores the epilogue of a zero product.  Grid: ceil(batch*m*n / 32) workgroups of 256.
constexpr int SPLITK_OUT = 32;
__global__ __launch_bounds__(256) void splitk_reduce(int m, int n, int batch, int splits, double alpha,
                                                     const double *__restrict__ part, GemmEpi ep,
                                                     double *__restrict__ C, int ldc, long sC) {
  __shared__ double red[8][SPLITK_OUT + 1], redo[8][SPLITK_OUT + 1];
  const long mn = (long)m * n, total = (long)batch * mn;
  const int o = threadIdx.x & (SPLITK_OUT - 1), g = threadIdx.x / SPLITK_OUT;
  const long e = (long)blockIdx.x * SPLITK_OUT + o;
  const int b = (int)(e / mn);
  const long r = e - b * mn;
  const int i = (int)(r / n), j = (int)(r - (long)i * n);
  double s = 0.0;
  if (e < total) {
#pragma unroll 4
    for (int q = g; q < splits; q += 8) s += part[(long)q * total + e];
  }
  red[g][o] = s;
  // the tail's outer products, shared by the groups like the splits
  redo[g][o] = ep.ext && e < total ? epi_outer(ep, b, i, j, g, 8) : 0.0;
  __syncthreads();
  if (g == 0 && e < total) {
    double t = red[0][o], u = redo[0][o];
#pragma unroll
    for (int h = 1; h < 8; ++h) {
      t += red[h][o];
      u += redo[h][o];
    }
    epi_store<true, true>(C + b * sC + (long)i * ldc + j, alpha * t, ep, b, i, j, u);
  }
}

// k == 1: an outer product.  One thread per output over the flattened (batch, row,
// column) index, with the product and epilogue of the MFMA path, which for k = 1 adds
// exact zeros to round(a b), so the results are the same bits at a fraction of the latency.
template <bool EXT>
__global__ __launch_bounds__(256) void rank1_kernel(int m, int n, int tA, int tB, double alpha,
                                                    const double *__restrict__ A, int lda, long sA,
                                                    const double *__restrict__ B, int ldb, long sB, GemmEpi ep,
                                                    double *__restrict__ C, int ldc, long sC, int batch) {
  const long mn = (long)m * n, e = blockIdx.x * 256L + threadIdx.x;
  if (e >= mn * batch) return;
  const int b = (int)(e / mn), r = (int)(e - b * mn), i = r / n, j = r - i * n;
  const double a = tA ? A[b * sA + i] : A[b * sA + (long)i * lda];
  const double bb = tB ? B[b * sB + (long)j * ldb] : B[b * sB + j];
  epi_store<EXT>(C + b * sC + (long)i * ldc + j, alpha * (a * bb), ep, b, i, j);
}

// n == 1: matrix-vector products.  One wave per output row: lanes stride over k, then a
// fixed-order wave reduction, so a row's value depends only on its own operands.
template <bool EXT>
__global__ __launch_bounds__(256) void gemv_kernel(int m, int k, int tA, int tB, double alpha,
                                                   const double *__restrict__ A, int lda, long sA,
                                                   const double *__restrict__ B, int ldb, long sB, GemmEpi ep,
                                                   double *__restrict__ C, int ldc, long sC, int batch) {
  const long o = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (o >= (long)batch * m) return;  // whole wave; no barriers below
  const int b = (int)(o / m), i = (int)(o - (long)b * m);
  const double *Ab = A + b * sA, *Bb = B + b * sB;
  double s = 0.0;
  for (int kk = lane; kk < k; kk += 64)
    s = fma(tA ? Ab[(long)kk * lda + i] : Ab[(long)i * lda + kk], tB ? Bb[kk] : Bb[(long)kk * ldb], s);
  s = gpx_wave_sum(s);
  if (lane == 0) epi_store<EXT>(C + b * sC + (long)i * ldc, alpha * s, ep, b, i, 0);
}

// ---------------------------------------------------------------------------
// Register-direct products.  One wave owns a (16 TM) x (16 TN) tile of C and feeds the matrix
// cores straight from global memory: no LDS staging, no barriers, every wave at its own pace.
// K advances in groups of 8; of a group, lane group g = lane / 16 supplies k = 2 g + s to MFMA
// step s = 0, 1 (the same permutation of k in both operands), so an operand whose rows run
// along k is read as one 16-byte load per lane and one whose rows run across k as 128-byte row
// segments.  The next group is in flight while the current one is multiplied.  Rows and columns
// past the edge re-read the last valid one (their results are not stored); a last partial group
// is masked to zero in both operands.  Large products are bound by the matrix cores, small ones
// by one launch and one round of loads.  Against tiles staged through LDS (64 x 64 or 32 x 32
// per workgroup), us: 20000 x 200 x 200, 4 products 245 -> 125 (26 -> 51 TF); 4001 x 256 x 256, 2
// 34 -> 29; 10000 x 6 x 1000 55 -> 17; 256^3, 2 9.6 -> 6.0; 100^3, 5 6.3 -> 4.3; 50^3 5.3 -> 4.1.
// ---------------------------------------------------------------------------
template <int TM, int TN, bool TA, bool TB, int KW, bool EXT>
__device__ __forceinline__ void gemm_direct_tile(int m, int n, int kbeg, int kend, double alpha, const double *A,
                                                 int lda, const double *B, int ldb, const GemmEpi &ep, double *C,
                                                 int ldc, int m0, int n0, int bidx, bool raw, double *red) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const GpxOperand<TM, !TA> oa(A, lda, m0, m, lane);
  const GpxOperand<TN, TB> ob(B, ldb, n0, n, lane);
  gpx_d4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = gpx_d4{0.0, 0.0, 0.0, 0.0};
  auto mul = [&](const GpxFrag<TM> &fa, const GpxFrag<TN> &fb) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = gpx_mfma16(fa.v[s][i], fb.v[s][j], acc[i][j]);
  };
  const int kw = KW > 1 ? wave : 0;
  const int groups = (kend - kbeg) >> 3, mine = (groups - kw + KW - 1) / KW;  // group kw + KW t of this wave
  const int kr = (kend - kbeg) & 7;
  const bool tail = kr && kw == groups % KW;
  constexpr bool EARLY = TM <= 2;  // registers to hold the tail from the start
  GpxFrag<EARLY ? TM : 1> ta;
  GpxFrag<EARLY ? TN : 1> tb;
  if constexpr (EARLY)
    if (tail) {
      oa.load_tail(ta, kbeg + 8 * groups, kr, lane);
      ob.load_tail(tb, kbeg + 8 * groups, kr, lane);
    }
  if (mine > 0) {
    constexpr int P = TM == 1 ? 4 : 2;  // groups in flight
    GpxFrag<TM> fa[P];
    GpxFrag<TN> fb[P];
    auto load = [&](int u, int t) {
      const int k0 = kbeg + 8 * (kw + KW * min(t, mine - 1));
      oa.load(fa[u], k0);
      ob.load(fb[u], k0);
    };
#pragma unroll
    for (int u = 0; u < P - 1; ++u) load(u, u);
    int t = 0;
    for (; t + P <= mine; t += P)
#pragma unroll
      for (int u = 0; u < P; ++u) {
        load((u + P - 1) % P, t + u + P - 1);
        mul(fa[u], fb[u]);
      }
#pragma unroll
    for (int u = 0; u < P - 1; ++u)
      if (t + u < mine) mul(fa[u], fb[u]);
  }
  if (tail) {
    if constexpr (EARLY) {
      mul(ta, tb);
    } else {
      GpxFrag<TM> fa;
      GpxFrag<TN> fb;
      oa.load_tail(fa, kbeg + 8 * groups, kr, lane);
      ob.load_tail(fb, kbeg + 8 * groups, kr, lane);
      mul(fa, fb);
    }
  }
  if constexpr (KW > 1) {
    // the waves' partial tiles, one row of 16 x 16 tiles at a time: wave r adds accumulator
    // register r (rows g + 4 r of each tile) of all four in wave order, and stores it
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (i) __syncthreads();
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[((wave * TN + j) * 4 + r) * 64 + lane] = acc[i][j][r];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int gm = m0 + i * 16 + (lane >> 4) + 4 * wave, gn = n0 + j * 16 + (lane & 15);
        double v = red[(j * 4 + wave) * 64 + lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) v += red[((w * TN + j) * 4 + wave) * 64 + lane];
        if (gm < m && gn < n) {
          double *c = C + (long)gm * ldc + gn;
          if (raw) *c = v;
          else epi_store<EXT>(c, alpha * v, ep, bidx, gm, gn);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + i * 16 + (lane >> 4) + 4 * r, gn = n0 + j * 16 + (lane & 15);
        if (gm < m && gn < n) {
          double *c = C + (long)gm * ldc + gn;
          if (raw) *c = acc[i][j][r];
          else epi_store<EXT>(c, alpha * acc[i][j][r], ep, bidx, gm, gn);
        }
      }
}

// Tiles are numbered column band fastest, then row band, then z = (batch, split).  KW = 1: the
// four waves of a workgroup take four consecutive tiles; KW = 4: they share one tile, each with
// every fourth group of K.  The n columns are cut into bands of ceil- or floor-balanced counts
// of 16-column tiles (n = 200: 4 + 3 + 3 + 3), so padding is below 16 columns in all.
// Workgroups are dealt to the XCDs in contiguous runs of tiles, which share operand panels.
template <int TM, int TX, bool TA, bool TB, int KW, bool EXT>
__global__ __launch_bounds__(256, 2) void gemm_direct_kernel(int m, int n, int k, double alpha, const double *__restrict__ A,
                                                          int lda, long sA, const double *__restrict__ B, int ldb,
                                                          long sB, GemmEpi ep, double *__restrict__ C, int ldc,
                                                          long sC, int batch, int splits, int kchunk,
                                                          double *__restrict__ part) {
  __shared__ double red[KW > 1 ? KW * TX * 256 : 1];
  const int nt = (n + 15) >> 4, cb = (nt + TX - 1) / TX, rb = (m + 16 * TM - 1) / (16 * TM);
  const long tiles = (long)rb * cb * batch * splits;
  const long chunk = gridDim.x >> 3, blk = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  long t = KW > 1 ? blk : blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= tiles) return;
  const int c = (int)(t % cb);
  t /= cb;
  const int r = (int)(t % rb), z = (int)(t / rb);
  const int b = z / splits, q = z % splits;
  const int lo = nt / cb, hi = nt % cb;  // the first `hi` bands have lo + 1 tiles
  const int tn = lo + (c < hi), n0 = 16 * (c * lo + min(c, hi)), m0 = 16 * TM * r;
  const int kbeg = q * kchunk, kend = min(k, kbeg + kchunk);
  A += b * sA;
  B += b * sB;
  const bool raw = part != nullptr;
  double *Cb = raw ? part + ((long)q * batch + b) * (long)m * n : C + b * sC;
  if (raw) ldc = n;
#define GEMM_TILE(TN)                                                                                               \
  gemm_direct_tile<TM, TN, TA, TB, KW, EXT>(m, n, kbeg, kend, alpha, A, lda, B, ldb, ep, Cb, ldc, m0, n0, b, raw, red)
  if constexpr (TX >= 4) {
    if (tn == 4) return GEMM_TILE(4);
    if (tn == 3) return GEMM_TILE(3);
  }
  if constexpr (TX >= 2)
    if (tn == 2) return GEMM_TILE(2);
  GEMM_TILE(1);
#undef GEMM_TILE
}

template <int TM, int KW, bool EXT>
int gemm_direct(int tA, int tB, int m, int n, int k, double alpha, const double *A, int lda, long sA, const double *B,
                int ldb, long sB, const GemmEpi &ep, double *C, int ldc, long sC, int batch, int splits, int kchunk,
                double *part, hipStream_t st) {
  const long cb = gpx_cdiv(gpx_cdiv(n, 16), TM), rb = gpx_cdiv(m, 16 * TM), tiles = rb * cb * batch * splits;
  const long blocks = KW > 1 ? tiles : (tiles + 3) / 4;
  const dim3 grid(8 * gpx_cdiv(blocks, 8));
#define GEMM_GO(TA, TB)                                                                                          \
  hipLaunchKernelGGL((gemm_direct_kernel<TM, TM, TA, TB, KW, EXT>), grid, dim3(256), 0, st, m, n, k, alpha, A, lda, sA, B, \
                     ldb, sB, ep, C, ldc, sC, batch, splits, kchunk, part)
  if (tA) {
    if (tB) GEMM_GO(true, true); else GEMM_GO(true, false);
  } else {
    if (tB) GEMM_GO(false, true); else GEMM_GO(false, false);
  }
#undef GEMM_GO
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// ---------------------------------------------------------------------------
// Weighted Gram matrices: out[d] = sum_n w_nd x_n x_n^T (+ gamma E[d]), symmetric, so only the
// 16 x 16 tiles on and above the diagonal are formed: pairs (r <= c) of column bands of at most
// four tiles (balanced, n = 200: 4 + 3 + 3 + 3), the weight applied to one operand's fragments
// as they arrive.  A workgroup owns one (pair, d, share of the points); its four waves take every
// fourth group of 8 points and are added in wave order.  Bound by the matrix cores (N = 20000,
// M = 200, 4 outputs: 84 us of which 47 are its products; a scaled copy of x and a full product
// took 45 + 317 us; N = 200, M = 50, 1 output 11 -> 9 us).
// ---------------------------------------------------------------------------
template <int TM, int TN, bool DIAG>
__device__ __forceinline__ void gram_tile(int N, int D, int M, int kbeg, int kend, const double *w, const double *X,
                                          int ldx, int m0, int n0, double *out, double *red) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4;
  const GpxOperand<TM, false> oa(X, ldx, m0, M, lane);
  const GpxOperand<TN, false> ob(X, ldx, n0, M, lane);
  gpx_d4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = gpx_d4{0.0, 0.0, 0.0, 0.0};
  auto mul = [&](const GpxFrag<TM> &fa, const GpxFrag<TN> &fb, const double *wv) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      double b[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = wv[s] * (DIAG ? fa.v[s][j] : fb.v[s][j]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = DIAG ? i : 0; j < TN; ++j) acc[i][j] = gpx_mfma16(fa.v[s][i], b[j], acc[i][j]);
    }
  };
  const int groups = (kend - kbeg) >> 3, mine = (groups - wave + 3) / 4;
  if (mine > 0) {
    GpxFrag<TM> fa[2];
    GpxFrag<TN> fb[2];
    double wv[2][2];
    auto load = [&](int u, int t) {
      const int k0 = kbeg + 8 * (wave + 4 * min(t, mine - 1));
      oa.load(fa[u], k0);
      if constexpr (!DIAG) ob.load(fb[u], k0);
      const double *wk = w + (long)k0 * D;
      wv[u][0] = wk[2L * g * D];
      wv[u][1] = wk[2L * g * D + D];
    };
    load(0, 0);
    int t = 0;
    for (; t + 2 <= mine; t += 2) {
      load(1, t + 1);
      mul(fa[0], fb[0], wv[0]);
      load(0, t + 2);
      mul(fa[1], fb[1], wv[1]);
    }
    if (t < mine) mul(fa[0], fb[0], wv[0]);
  }
  const int kr = (kend - kbeg) & 7;
  if (kr && wave == groups % 4) {
    const int k0 = kbeg + 8 * groups;
    GpxFrag<TM> fa;
    GpxFrag<TN> fb;
    oa.load_tail(fa, k0, kr, lane);
    ob.load_tail(fb, k0, kr, lane);
    double wv[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) wv[s] = 2 * g + s < kr ? w[(long)(k0 + 2 * g + s) * D] : 0.0;
    mul(fa, fb, wv);
  }
  // the waves' partial tiles, one row of 16 x 16 tiles at a time: wave r adds accumulator
  // register r of all four in wave order, and stores it
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int j = DIAG ? i : 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave * TN + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int j = DIAG ? i : 0; j < TN; ++j) {
      const int gm = m0 + i * 16 + g + 4 * wave, gn = n0 + j * 16 + (lane & 15);
      double v = red[(j * 4 + wave) * 64 + lane];
#pragma unroll
      for (int u = 1; u < 4; ++u) v += red[((u * TN + j) * 4 + wave) * 64 + lane];
      if (gm < M && gn < M) out[(long)gm * M + gn] = v;
    }
  }
}

// Grid: (splits, pairs, D), largest pairs (lowest bands) first.
__global__ __launch_bounds__(256, 2) void gram_kernel(int N, int D, int M, int kchunk, const double *__restrict__ w,
                                                      const double *__restrict__ X, int ldx, double *__restrict__ part) {
  __shared__ double red[16 * 256];
  const int nt = (M + 15) >> 4, cb = (nt + 3) / 4, lo = nt / cb, hi = nt % cb, d = blockIdx.z;
  int r = 0, c = blockIdx.y;
  while (c >= cb - r) {  // pair index -> (r, r + c)
    c -= cb - r;
    ++r;
  }
  c += r;
  const int tm = lo + (r < hi), tn = lo + (c < hi), m0 = 16 * (r * lo + min(r, hi)), n0 = 16 * (c * lo + min(c, hi));
  const int kbeg = blockIdx.x * kchunk, kend = min(N, kbeg + kchunk);
  double *out = part + ((long)blockIdx.x * D + d) * M * M;
#define GRAM_TILE(TM, TN, DIAG) gram_tile<TM, TN, DIAG>(N, D, M, kbeg, kend, w + d, X, ldx, m0, n0, out, red)
  if (r == c) {
    if (tm == 4) GRAM_TILE(4, 4, true);
    else if (tm == 3) GRAM_TILE(3, 3, true);
    else if (tm == 2) GRAM_TILE(2, 2, true);
    else GRAM_TILE(1, 1, true);
  } else if (tm == 4) {
    if (tn == 4) GRAM_TILE(4, 4, false); else GRAM_TILE(4, 3, false);
  } else {  // two bands or more: at least 3 + 2 tiles
    if (tn == 3) GRAM_TILE(3, 3, false); else GRAM_TILE(3, 2, false);
  }
#undef GRAM_TILE
}

// Sum of the partial Gram matrices over the splits (fixed order) for i <= j, stored at (i, j)
// and (j, i); same thread layout as splitk_reduce.
__global__ __launch_bounds__(256) void gram_reduce(int D, int M, int splits, const double *__restrict__ part,
                                                   GemmEpi ep, double *__restrict__ out) {
  __shared__ double red[8][SPLITK_OUT + 1];
  const long mm = (long)M * M, total = mm * D;
  const int o = threadIdx.x & (SPLITK_OUT - 1), g = threadIdx.x / SPLITK_OUT;
  const long e = (long)blockIdx.x * SPLITK_OUT + o;
  const int b = (int)(e / mm), r = (int)(e - b * mm), i = r / M, j = r - i * M;
  const bool on = e < total && i <= j;
  double s = 0.0;
  if (on) {
#pragma unroll 4
    for (int q = g; q < splits; q += 8) s += part[(long)q * total + e];
  }
  red[g][o] = s;
  __syncthreads();
  if (g == 0 && on) {
    double t = red[0][o];
#pragma unroll
    for (int h = 1; h < 8; ++h) t += red[h][o];
    out += b * mm;
    epi_store<true>(out + (long)i * M + j, t, ep, b, i, j);
    if (i != j) epi_store<true>(out + (long)j * M + i, t, ep, b, j, i);
  }
}

}  // namespace

extern "C" {

long gpx_gram_workspace(int D, int M, int splits) { return (long)splits * D * M * M; }

int gpx_gram(int N, int D, int M, const double *w, const double *X, int ldx, double gamma, const double *E,
             long strideE, double *out, int splits, double *work, void *stream) {
  if (N < 0 || D < 0 || M < 0 || splits < 1 || D > 65535) return GPX_EINVAL;
  if (E && strideE < 0) return GPX_EINVAL;
  if (D == 0 || M == 0) return GPX_OK;
  if (!out || (N > 0 && (!w || !X || !work || ldx < M))) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  int kchunk = (N + splits - 1) / splits;
  kchunk = (kchunk + 7) / 8 * 8;
  splits = kchunk ? (N + kchunk - 1) / kchunk : 0;
  const GemmEpi ep{0.0, gamma, E, M, strideE, 0, M, M, GpxGemmTail{}};
  if (splits) {
    const int cb = (int)gpx_cdiv(gpx_cdiv(M, 16), 4);
    if ((long)cb * (cb + 1) / 2 > 65535) return GPX_ETOOBIG;
    hipLaunchKernelGGL(gram_kernel, dim3(splits, cb * (cb + 1) / 2, D), dim3(256), 0, st, N, D, M, kchunk, w, X, ldx,
                       work);
    GPX_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(gram_reduce, dim3(gpx_cdiv((long)D * M * M, SPLITK_OUT)), dim3(256), 0, st, D, M, splits,
                     (const double *)work, ep, out);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// Workspace (doubles) that gpx_gemm_batched needs for a given split count.
long gpx_gemm_workspace(int m, int n, int batch, int splits) {
  return splits > 1 ? (long)splits * batch * m * n : 0;
}

int gpx_gemm_batched_tail(int transA, int transB, int m, int n, int k, double alpha,
                        const double *A, int lda, long strideA,
                        const double *B, int ldb, long strideB,
                        double beta, double *C, int ldc, long strideC,
                        double gamma, const double *E, int ldE, long strideE, const GpxGemmTail *tail,
                        int batch, int splits, double *work, int tile, void *stream) {
  if (m < 0 || n < 0 || k < 0 || batch < 0 || splits < 1) return GPX_EINVAL;
  if (E && (ldE < n || strideE < 0)) return GPX_EINVAL;
  GemmEpi ep{beta, gamma, E, ldE, strideE, tail != nullptr, m, n, tail ? *tail : GpxGemmTail{}};
  if (m == 0 || n == 0 || batch == 0) return GPX_OK;
  if (!A || !B || !C) return GPX_EINVAL;
  if (tail && (tail->terms < 0 || (tail->terms && (!tail->U || !tail->V)))) return GPX_EINVAL;
  if (splits > 1 && !work) return GPX_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (k == 0) {  // C = beta * C
    hipLaunchKernelGGL(splitk_reduce, dim3(gpx_cdiv((long)batch * m * n, SPLITK_OUT)), dim3(256), 0, st, m, n, batch,
                       0, 0.0, (const double *)nullptr, ep, C, ldc, strideC);
    GPX_CHECK_LAUNCH();
    return GPX_OK;
  }
  // outer products and matrix-vector products (automatic tile choice only)
  if (tile == 0 && splits == 1 && k == 1) {
    if (tail)
      hipLaunchKernelGGL(rank1_kernel<true>, dim3(gpx_cdiv((long)batch * m * n, 256)), dim3(256), 0, st, m, n, transA,
                       transB, alpha, A, lda, strideA, B, ldb, strideB, ep, C, ldc, strideC, batch);
    else
      hipLaunchKernelGGL(rank1_kernel<false>, dim3(gpx_cdiv((long)batch * m * n, 256)), dim3(256), 0, st, m, n, transA,
                       transB, alpha, A, lda, strideA, B, ldb, strideB, ep, C, ldc, strideC, batch);
    GPX_CHECK_LAUNCH();
    return GPX_OK;
  }
  if (tile == 0 && splits == 1 && n == 1) {
    if (tail)
      hipLaunchKernelGGL(gemv_kernel<true>, dim3(gpx_cdiv((long)batch * m, 4)), dim3(256), 0, st, m, k, transA, transB,
                       alpha, A, lda, strideA, B, ldb, strideB, ep, C, ldc, strideC, batch);
    else
      hipLaunchKernelGGL(gemv_kernel<false>, dim3(gpx_cdiv((long)batch * m, 4)), dim3(256), 0, st, m, k, transA, transB,
                       alpha, A, lda, strideA, B, ldb, strideB, ep, C, ldc, strideC, batch);
    GPX_CHECK_LAUNCH();
    return GPX_OK;
  }
  int kchunk = (k + splits - 1) / splits;
  kchunk = (kchunk + 7) / 8 * 8;
  splits = (k + kchunk - 1) / kchunk;
  double *part = splits > 1 ? work : nullptr;
  if ((long)batch * splits > 65535L) return GPX_EINVAL;
  const long z = (long)batch * splits, t4 = z * gpx_cdiv(m, 64) * gpx_cdiv(n, 64),
             t2 = z * gpx_cdiv(m, 32) * gpx_cdiv(n, 32), t1 = z * gpx_cdiv(m, 16) * gpx_cdiv(n, 16);
  int rc;
#define GEMM_DIRECT1(TM, KW, EXT)                                                                                 \
  gemm_direct<TM, KW, EXT>(transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, ep, C, ldc, strideC, \
                           batch, splits, kchunk, part, st)
#define GEMM_DIRECT(TM, KW) tail ? GEMM_DIRECT1(TM, KW, (TM < 4)) : GEMM_DIRECT1(TM, KW, false)
  // (with a tail never 64 x 64 per wave: its 64 stores per lane each carry the epilogue)
  // 64 x 64 per wave once there are two such tiles per SIMD (20000 x n x n, 4 products, us
  // against 32 x 32: n = 256 172 : 228, 200 125 : 133, 128 (2504 tiles) 63 : 65; 5000 x 100 x 100, 4
  // (632 tiles) 24 : 18).  16 x 16 per workgroup, its waves sharing k, where those are at most three
  // per CU (against 32 x 32: 128^3 4.4 : 5.5, 200^3, 4 (676 tiles) 5.8 : 6.0, 128^3, 32 (2048) 13 : 7.8).
  // Else 32 x 32: a tile per wave takes whole rounds of 1024 (a wave per SIMD), four waves sharing
  // a tile's k take rounds of 256 at a quarter of the time and 3% more, and four more waves' loads in
  // flight.  So a tile per wave where its rounds are at least 7/8 full (us against shared k, 256 x 256
  // x 256 or x 256 x 256 (tiles): (768) 16.4 : 14.1, (896) 16.7 : 17.3, (1008) 16.9 : 17.4, (1256) 27.8 : 20.4,
  // (1504) 28.3 : 23.9, (2000) 29.3 : 30.0, (4000) 51.8 : 54.2; n = k = 100: (1252) 13.6 : 11.3, (1920) 14.1 :
  // 15.2), 3/4 where k is short (64^3 (800) 8.6 : 9.1, (1600) 13.1 : 13.9; 50^3 (1200) 10.2 : 9.3, (1600) 10.6 : 11.5),
  // and k is not so long that the loads decide (200 x 1000 (882) 48 : 41, (2625) 113 : 100).  Up to
  // k = 16 most of four waves have nothing to share, and only few tiles gain from them (k = 8 (658) 5.9 :
  // 6.0, (1256) 7.0 : 7.8; k = 12 (504) 6.1 : 5.7, (752) 6.4 : 6.4; k = 32 (512) 7.0 : 6.0, (1256) 9.4 : 8.6).
  const bool full = t2 >= 4096 || 8 * t2 > (k <= 64 ? 6 : 7) * 1024 * (long)gpx_cdiv(t2, 1024);
  if (!tail && (tile == 64 || (tile != 32 && t4 >= 2048 && k >= 64))) rc = GEMM_DIRECT(4, 1);
  else if (tile != 32 && t1 <= 768) rc = GEMM_DIRECT(1, 4);
  else if (k <= 16 ? t2 > 576 : k <= 256 && full) rc = GEMM_DIRECT(2, 1);
  else rc = GEMM_DIRECT(2, 4);
#undef GEMM_DIRECT
#undef GEMM_DIRECT1
  if (rc != GPX_OK) return rc;
  if (part) {
    const long total = (long)batch * m * n;
    hipLaunchKernelGGL(splitk_reduce, dim3(gpx_cdiv(total, SPLITK_OUT)), dim3(256), 0, st, m, n, batch, splits, alpha,
                       (const double *)part, ep, C, ldc, strideC);
    GPX_CHECK_LAUNCH();
  }
  return GPX_OK;
}

int gpx_gemm_batched_ex(int transA, int transB, int m, int n, int k, double alpha,
                        const double *A, int lda, long strideA,
                        const double *B, int ldb, long strideB,
                        double beta, double *C, int ldc, long strideC,
                        double gamma, const double *E, int ldE, long strideE,
                        int batch, int splits, double *work, int tile, void *stream) {
  return gpx_gemm_batched_tail(transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc,
                               strideC, gamma, E, ldE, strideE, nullptr, batch, splits, work, tile, stream);
}

int gpx_gemm_batched(int transA, int transB, int m, int n, int k, double alpha,
                     const double *A, int lda, long strideA,
                     const double *B, int ldb, long strideB,
                     double beta, double *C, int ldc, long strideC,
                     int batch, int splits, double *work, int tile, void *stream) {
  return gpx_gemm_batched_ex(transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc,
                             strideC, 0.0, nullptr, 0, 0, batch, splits, work, tile, stream);
}

}  // extern "C"
