// Grouped predictive mean / variance for many resident models in one launch.
//
// One workgroup (8 waves) per work item = up to SERVE_TILE query points of one request
// against one model.  Each model is a chain of at most two sparse-GP layers in posterior form:
//   deterministic inputs (first layer): kfu = SE(x, Z), m = kfu A^T,
//       v = sf2 + kfu B_det kfu^T                      (base_models.py:265-284)
//   Gaussian inputs (second layer):      m = psi1 A^T,
//       v = sf2 + <B_sto, psi2> - m^2                   (base_models.py:286-307)
// Both quadratic forms run on the matrix cores with the 16 points as MFMA columns; psi2 is
// never stored.  Every per-point reduction runs in a fixed order, independent of the other
// points of the launch, so a query's result is bitwise the same alone or batched with any
// other requests.
//
// What bounds it: the FP64 matrix cores for the first layer (M^2/4 MFMA columns per output,
// B_det streamed from the L2 once per item) and the exps of psi2 for the second (16 M (M+1)/2
// of them per item, about 56 FP64 vector instructions per 4).  Forming 1/l and the log
// factors per (point, inducing point, dimension), the psi2 features per entry and the B_det
// contraction one column per thread were most of the earlier kernel's time.  One request of
// one point, wall microseconds, before -> now: two layers of M = 256, Din 8, hidden 5 1296 ->
// 287; M = 64, Din 10 217 -> 91; one layer of M = 128 101 -> 71 (70 of it host and copies); 24
// requests of 1-4096 points over 32 models of M 32-256: the launch 1816 -> 411.
#include "gpx_common.h"

#define SERVE_TILE 16
#define SERVE_MMAX 256
#define SERVE_QMAX 16
#define SERVE_HMAX 8

struct GpxServeLayer {
  int type;  // 0: deterministic inputs, 1: Gaussian inputs
  int M, Din, Dout;
  const double *zu, *ls, *sf;
  const double *A;  // Dout x M
  const double *B;  // Dout x M x M
};

struct GpxServeModel {
  int nlayers;
  int Din, Dout;
  int pad_;
  const double *sn;  // log noise std for predict_y (may be NULL)
  GpxServeLayer layer[2];
};

struct GpxServeItem {
  int model;
  int rows;
  long in_off;   // doubles into X (rows x Din)
  long out_off;  // doubles into mean / var (rows x Dout)
};

namespace {

constexpr int SV_NW = 8;                  // waves per workgroup
constexpr int SV_NT = 64 * SV_NW;
constexpr int SV_DCH = 8;                 // outputs of a deterministic layer per pass
constexpr int SV_ZS = SERVE_QMAX + 1;

// 79 KB, so two workgroups share a CU.
struct ServeLds {
  union {
    double zs[SERVE_MMAX * SV_ZS];        // Z, rows of SV_ZS (columns past Q zero)
    // sums over the waves, once Z is done with: [job][point], jobs = (output, row tile) of the
    // first layer or (wave, output) of the second
    struct {
      double pv[SV_DCH * 16][SERVE_TILE], pm[SV_DCH * 16][SERVE_TILE];
    };
  };
  double ft[SERVE_MMAX * SERVE_TILE];     // [m][point]: kfu (first layer) or u (second)
  double xin[SERVE_TILE][SERVE_QMAX];     // inputs
  double hm[SERVE_TILE][SERVE_HMAX], hv[SERVE_TILE][SERVE_HMAX];
  double il[SERVE_QMAX];                  // 1 / l
  double pd[SERVE_TILE][SERVE_HMAX], pw[SERVE_TILE][SERVE_HMAX];  // psi2: d, w
  double p1[SERVE_TILE][SERVE_HMAX];                              // psi1: 1 / (2 (l + v))
  double c1[SERVE_TILE][SERVE_HMAX], c2[SERVE_TILE][SERVE_HMAX];  // their log factors
  double etab[32];
};

// v + the same point's values in the other three 16-lane rows.
__device__ __forceinline__ double rows_sum(double v) { return gpx_swap_add<32>(gpx_swap_add<16>(v)); }

// Lane R of each 16-lane row to the whole row.
template <int R>
__device__ __forceinline__ double row_bcast(double v) {
  return __longlong_as_double(
      __builtin_amdgcn_mov_dpp((long long)__double_as_longlong(v), 0x150 + R, 0xF, 0xF, true));
}

// <B_sto[d], psi2> over the wave's rows a of every tile, for the 16 points: with
// u_ma = sum_q [log(l d)/4 - d (mu-z)^2/2] and w = v d/(2 l) the psi2 exponent is
// u_a + u_b - sum_q w (z_aq - z_bq)^2 (KS slices of 4), as in the fused training kernels.
// Tiles (A < B) carry B_ab + B_ba, diagonal tiles B_ab.  ONE: a single output, per-lane FMAs
// (acc[0] of lane (b, point)); otherwise the MFMA contraction (acc[r] = output lane/16 + 4r).
template <int KS, bool ONE>
__device__ __forceinline__ gpx_d4 serve_psi2(const ServeLds &sm, const GpxServeLayer &L, int lane, int wave) {
  const int M = L.M, T = (M + 15) / 16, ka = lane & 15, kq = lane >> 4;
  double bf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) bf[s] = sm.pw[ka][kq + 4 * s];
  gpx_d4 acc = gpx_d4{0.0, 0.0, 0.0, 0.0};
  const int d = ONE ? 0 : min(ka, L.Dout - 1);
  const double *Bd = L.B + (long)d * M * M;
  for (int B = 0; B < T; ++B) {
    const int jl = min(16 * B + ka, M - 1);
    double zb[KS], ub[4];
#pragma unroll
    for (int s = 0; s < KS; ++s) zb[s] = sm.zs[jl * SV_ZS + kq + 4 * s];
#pragma unroll
    for (int r = 0; r < 4; ++r) ub[r] = sm.ft[(16 * B + kq + 4 * r) * SERVE_TILE + ka];
    // rows a = wave, wave + 8, ... up to the end of tile B; B_sto is loaded PF rows ahead (at
    // clamped rows, so every load is in bounds; one row ahead with four loads each for B_ab and
    // B_ba left the two-layer M = 256 request at 328).  ONE: lane (kq, j = ka % 4) loads b = kq + 4j,
    // one load per row for the four b of its lane row, spread by row broadcasts below.
    const int na = min(16 * (B + 1), M);
    constexpr int NB = ONE ? 1 : 4, PF = ONE ? 4 : 1;
    double bn[PF][NB], cn[PF][NB];
    auto load = [&](int a, int i) {
      const int al = min(a, na - 1);
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        const int b = min(16 * B + kq + 4 * (ONE ? (ka & 3) : r), M - 1);
        bn[i][r] = Bd[(long)al * M + b];
        cn[i][r] = Bd[(long)b * M + al];
      }
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) load(wave + SV_NW * i, i);
    for (int a0 = wave; a0 < na; a0 += SV_NW * PF) {
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        const int a = a0 + SV_NW * i;
        if (a >= na) break;  // wave-uniform
        double bs[4];
        const bool off = a < 16 * B;
#pragma unroll
        for (int r = 0; r < NB; ++r) bs[r] = off ? bn[i][r] + cn[i][r] : bn[i][r];
        load(a + SV_NW * PF, i);
        if constexpr (ONE) {
          const double t = bs[0];
          bs[0] = row_bcast<0>(t);
          bs[1] = row_bcast<1>(t);
          bs[2] = row_bcast<2>(t);
          bs[3] = row_bcast<3>(t);
        }
        const double ua = sm.ft[a * SERVE_TILE + ka];
        gpx_d4 e;
#pragma unroll
        for (int r = 0; r < 4; ++r) e[r] = ua + ub[r];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const double dz = sm.zs[a * SV_ZS + kq + 4 * s] - zb[s];
          e = gpx_mfma16(-dz * dz, bf[s], e);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double p = gpx_exp_tab(e[r], sm.etab);
          if constexpr (ONE) acc[0] = fma(bs[r], p, acc[0]);
          else acc = gpx_mfma16(bs[r], p, acc);
        }
      }
    }
  }
  return acc;
}

__global__ __launch_bounds__(SV_NT, 4) void serve_kernel(const GpxServeModel *__restrict__ models,
                                                      const GpxServeItem *__restrict__ items,
                                                      const double *__restrict__ X,
                                                      double *__restrict__ mean, double *__restrict__ var,
                                                      int noisy) {
  __shared__ ServeLds sm;
  const GpxServeItem it = items[blockIdx.x];
  const GpxServeModel &mod = models[it.model];
  const int tid = threadIdx.x, rows = it.rows, lane = tid & 63, ka = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  gpx_exp_table_init(sm.etab);
  for (int e = tid; e < SERVE_TILE * mod.Din; e += SV_NT) {
    const int p = e / mod.Din, q = e % mod.Din;
    sm.xin[p][q] = (p < rows) ? X[it.in_off + (long)p * mod.Din + q] : 0.0;
  }
  const double sn2 = (noisy && mod.sn) ? exp(2.0 * mod.sn[0]) : 0.0;
  for (int l = 0; l < mod.nlayers; ++l) {
    const GpxServeLayer &L = mod.layer[l];
    const int M = L.M, Q = L.Din, T = (M + 15) / 16;
    const double sf2 = exp(2.0 * L.sf[0]);
    const bool last = (l == mod.nlayers - 1);
    // hyper-parameters, inducing inputs and (second layer) the points' constants
    if (tid < SERVE_QMAX) sm.il[tid] = tid < Q ? exp(-2.0 * L.ls[tid]) : 0.0;
    {
      const int ZQ = 4 * ((Q + 3) / 4);
      for (int e = tid; e < M * ZQ; e += SV_NT) {
        const int m = e / ZQ, q = e % ZQ;
        sm.zs[m * SV_ZS + q] = q < Q ? L.zu[m * Q + q] : 0.0;
      }
    }
    if (L.type == 1 && tid < SERVE_TILE * SERVE_HMAX) {
      const int p = tid / SERVE_HMAX, q = tid % SERVE_HMAX;
      const bool in = q < Q;
      const double l2 = in ? exp(2.0 * L.ls[q]) : 1.0, v = in ? sm.hv[p][q] : 0.0;
      const double d = 1.0 / (2.0 * v + l2), e1 = 1.0 / (v + l2);
      sm.pd[p][q] = d;
      sm.pw[p][q] = 0.5 * v * d / l2;
      sm.p1[p][q] = 0.5 * e1;
      sm.c1[p][q] = 0.5 * log(l2 * e1);
      sm.c2[p][q] = 0.25 * log(l2 * d);
    }
    __syncthreads();
    const int p = tid & 15;  // this thread's point in the feature loops (m = tid / 16 + 32 j)
    if (L.type == 0) {
      for (int m = tid >> 4; m < 16 * T; m += SV_NT / 16) {
        double acc = 0.0;
        const double *zm = sm.zs + min(m, M - 1) * SV_ZS;
        for (int q = 0; q < Q; ++q) {
          const double dz = sm.xin[p][q] - zm[q];
          acc = fma(dz * sm.il[q], dz, acc);
        }
        sm.ft[m * SERVE_TILE + p] = m < M ? sf2 * exp(-0.5 * acc) : 0.0;
      }
      __syncthreads();
      // jobs (output d, row tile I) dealt to the waves: W_b = sum_a B_d[a][b] k_a for the 16
      // rows b of the tile, then sum_b k_b W_b and sum_b k_b A_db
      for (int d0 = 0; d0 < L.Dout; d0 += SV_DCH) {
        const int nd = min(SV_DCH, L.Dout - d0);
        for (int j = wave; j < nd * T; j += SV_NW) {
          const int d = d0 + j / T, I = j % T, bl = min(16 * I + ka, M - 1);
          const double *Bc = L.B + (long)d * M * M + bl;
          gpx_d4 w = gpx_d4{0.0, 0.0, 0.0, 0.0};
          constexpr int U = 8;  // k-slices per step; the next step's B loaded ahead
          double an[U];
          auto load = [&](int k0) {
#pragma unroll
            for (int s = 0; s < U; ++s) an[s] = Bc[(long)min(k0 + 4 * s + kq, M - 1) * M];
          };
          load(0);
          for (int k0 = 0; k0 < M; k0 += 4 * U) {
            double av[U];
#pragma unroll
            for (int s = 0; s < U; ++s) av[s] = an[s];
            load(k0 + 4 * U);
#pragma unroll
            for (int s = 0; s < U; ++s)
              if (k0 + 4 * s < M) w = gpx_mfma16(av[s], sm.ft[(k0 + 4 * s + kq) * SERVE_TILE + ka], w);
          }
          double vq = 0.0, vm = 0.0;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int b = 16 * I + kq + 4 * r;
            const double f = sm.ft[b * SERVE_TILE + ka];  // 0 past M
            vq = fma(f, w[r], vq);
            vm = fma(f, L.A[(long)d * M + min(b, M - 1)], vm);
          }
          vq = rows_sum(vq);
          vm = rows_sum(vm);
          if (kq == 0) {
            sm.pv[j][ka] = vq;
            sm.pm[j][ka] = vm;
          }
        }
        __syncthreads();
        if (tid < nd * SERVE_TILE) {
          const int dd = tid / SERVE_TILE, d = d0 + dd;
          double m = 0.0, v = 0.0;
          for (int I = 0; I < T; ++I) {
            m += sm.pm[dd * T + I][p];
            v += sm.pv[dd * T + I][p];
          }
          v += sf2;
          if (last) {
            if (p < rows) {
              mean[it.out_off + (long)p * L.Dout + d] = m;
              var[it.out_off + (long)p * L.Dout + d] = v + sn2;
            }
          } else {
            sm.hm[p][d] = m;
            sm.hv[p][d] = v;
          }
        }
        __syncthreads();
      }
    } else {
      // u of every inducing point
      double cc1 = 0.0, cc2 = 0.0;
      for (int q = 0; q < Q; ++q) {
        cc1 += sm.c1[p][q];
        cc2 += sm.c2[p][q];
      }
      for (int m = tid >> 4; m < 16 * T; m += SV_NT / 16) {
        double u = cc2;
        const double *zm = sm.zs + min(m, M - 1) * SV_ZS;
        for (int q = 0; q < Q; ++q) {
          const double dz = sm.hm[p][q] - zm[q];
          u = fma(-0.5 * sm.pd[p][q] * dz, dz, u);
        }
        // no lower than the padding's: psi2 is an exact 0 there, and an exponent of any size stays
        // within what gpx_exp_tab reduces (a NaN stays)
        sm.ft[m * SERVE_TILE + p] = m < M && !(u < -1.0e4) ? u : -1.0e4;
      }
      __syncthreads();
      gpx_d4 acc;
      const bool one = L.Dout == 1;
      if (Q <= 4) acc = one ? serve_psi2<1, true>(sm, L, lane, wave) : serve_psi2<1, false>(sm, L, lane, wave);
      else acc = one ? serve_psi2<2, true>(sm, L, lane, wave) : serve_psi2<2, false>(sm, L, lane, wave);
      // the mean, sum_m psi1_m A_dm over this thread's m (d < 16, this wave's four rows of
      // lanes and then the waves in order)
      double vm[16];
#pragma unroll
      for (int d = 0; d < 16; ++d) vm[d] = 0.0;
      for (int m = tid >> 4; m < M; m += SV_NT / 16) {
        double e1 = cc1;
        const double *zm = sm.zs + m * SV_ZS;
        for (int q = 0; q < Q; ++q) {
          const double dz = sm.hm[p][q] - zm[q];
          e1 = fma(-sm.p1[p][q] * dz, dz, e1);
        }
        const double psi1 = sf2 * exp(e1);
        vm[0] = fma(psi1, L.A[m], vm[0]);
        if (!one) {
#pragma unroll
          for (int d = 1; d < 16; ++d)
            if (d < L.Dout) vm[d] = fma(psi1, L.A[(long)d * M + m], vm[d]);
        }
      }
      __syncthreads();  // pv, pm overlay Z
      if (one) {
        const double t = rows_sum(vm[0]), v = rows_sum(acc[0]);
        if (kq == 0) {
          sm.pm[wave * 16][ka] = t;
          sm.pv[wave * 16][ka] = v;
        }
      } else {
#pragma unroll
        for (int d = 0; d < 16; ++d) {
          const double t = rows_sum(vm[d]);
          if (kq == 0) sm.pm[wave * 16 + d][ka] = t;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) sm.pv[wave * 16 + kq + 4 * r][ka] = acc[r];
      }
      __syncthreads();
      if (tid < L.Dout * SERVE_TILE) {
        const int d = tid / SERVE_TILE;
        double m = 0.0, v = 0.0;
#pragma unroll
        for (int w = 0; w < SV_NW; ++w) {
          m += sm.pm[w * 16 + d][p];
          v += sm.pv[w * 16 + d][p];
        }
        v = sf2 + sf2 * sf2 * v - m * m;
        if (last) {
          if (p < rows) {
            mean[it.out_off + (long)p * L.Dout + d] = m;
            var[it.out_off + (long)p * L.Dout + d] = v + sn2;
          }
        } else {
          sm.hm[p][d] = m;
          sm.hv[p][d] = v;
        }
      }
      __syncthreads();
    }
  }
}

}  // namespace

extern "C" {

int gpx_serve_tile(void) { return SERVE_TILE; }
int gpx_serve_desc_sizes(int *model_bytes, int *item_bytes) {
  if (!model_bytes || !item_bytes) return GPX_EINVAL;
  *model_bytes = (int)sizeof(GpxServeModel);
  *item_bytes = (int)sizeof(GpxServeItem);
  return GPX_OK;
}

// One launch over `nitems` work items (each <= SERVE_TILE rows of one request).  Models
// need M <= 256, layer inputs <= 16 dims, hidden width <= 8; the caller validates the
// descriptor tables (gpx_serve_validate) when it builds them.
int gpx_predict_grouped(int nitems, const void *models, const void *items, const double *X,
                        double *mean, double *var, int noisy, void *stream) {
  if (nitems < 0 || !models || !items || !X || !mean || !var) return GPX_EINVAL;
  if (nitems == 0) return GPX_OK;
  hipLaunchKernelGGL(serve_kernel, dim3(nitems), dim3(SV_NT), 0, (hipStream_t)stream,
                     (const GpxServeModel *)models, (const GpxServeItem *)items, X, mean, var, noisy);
  GPX_CHECK_LAUNCH();
  return GPX_OK;
}

// Host-side check of one model descriptor (host copy) against the kernel's limits.
int gpx_serve_validate(const void *model) {
  const GpxServeModel *m = (const GpxServeModel *)model;
  if (!m || m->nlayers < 1 || m->nlayers > 2) return GPX_EINVAL;
  if (m->Din < 1 || m->Din > SERVE_QMAX) return GPX_EINVAL;
  int din = m->Din;
  for (int l = 0; l < m->nlayers; ++l) {
    const GpxServeLayer &L = m->layer[l];
    if (L.type != (l == 0 ? 0 : 1)) return GPX_EINVAL;
    if (L.M < 1 || L.M > SERVE_MMAX || L.Din != din || L.Dout < 1) return GPX_EINVAL;
    if (l < m->nlayers - 1 && L.Dout > SERVE_HMAX) return GPX_EINVAL;
    if (L.type == 1 && L.Dout > 16) return GPX_EINVAL;  // one 16-row MFMA tile of outputs
    if (!L.zu || !L.ls || !L.sf || !L.A || !L.B) return GPX_EINVAL;
    din = L.Dout;
  }
  if (din != m->Dout) return GPX_EINVAL;
  return GPX_OK;
}

}  // extern "C"
