// hyper.hip -- FP64 hyperprior statistics, adaptive noise, evaluation, RNG
// probes.
//
// Normal-Wishart conjugate update (CondNormalWishart, mvnormal.cpp:314-336):
//   mu_c = (kappa mu0 + sum U) / (kappa + N),  kappa_c = kappa + N,
//   nu_c = nu + N,  X = T + U U^T + kappa mu0 mu0^T - kappa_c mu_c mu_c^T,
//   T_c = X^{-1};  Lambda ~ Wishart(T_c, nu_c) by Bartlett
//   (mvnormal.cpp:217-266);  mu ~ N(mu_c, (kappa_c Lambda)^{-1})
//   (MvNormal_prec, mvnormal.cpp:169-184).
// The sufficient statistics are accumulated over columns by many work-groups
// in FP64 and reduced in place into the first partial row, beside work-groups
// that make the draw's random numbers (which need no statistics); the K x K
// draw then runs in one work-group (nwdraw.hip).
#include "common.h"
#include "kernels.h"

namespace mgpu {

constexpr int kMaxStatBlocks = 512;

int hyper_stats_blocks(int N) {
  int b = (N + 127) / 128;
  if (b < 1) b = 1;
  if (b > kMaxStatBlocks) b = kMaxStatBlocks;
  return b;
}

template <int KP>
struct StatShape {
  static constexpr int TD = KP / 4;                       // 4 x 4 tiles per dimension
  static constexpr int GT = TD * TD < 64 ? 64 : TD * TD;  // threads per column group
  static constexpr int G = GT >= 256 ? 1 : 256 / GT;      // column groups per block
  static constexpr int THREADS = GT * G;
  static constexpr int TC = 16;                           // columns per LDS tile
  static constexpr int EPT = TC * KP / GT;                // tile elements loaded per thread
  static constexpr int TILE = G * 2 * TC * KP;            // doubles, double buffered
  static constexpr int RED = G > 1 ? G * (KP + KP * KP) : 0;
  static constexpr int SMEM = TILE > RED ? TILE : RED;
};

// Sufficient statistics of x_n = U[:, n] - sub[:, n] (sub optional, FP32,
// same ld) over the block's run of columns, in FP64:
//   partial[blk] = (sum_n x_n (K), sum_n x_n x_n^T (K x K, col-major)).
// The block's columns are split between G column groups; each group streams
// its columns through a double-buffered LDS tile of 16 columns (the loads of
// tile t + 1 are in flight while tile t is used), and thread (ti, tj) of a
// group owns rows 4ti..4ti+3 x columns 4tj..4tj+3 of the K x K sum in
// registers.  The groups' sums are combined in group order.
template <typename T, int KP>
__global__ void __launch_bounds__(StatShape<KP>::THREADS)
    k_hyper_stats(const T* __restrict__ U, const float* __restrict__ sub, int ld, int N, int K, int cols,
                  double* __restrict__ partial) {
  using S = StatShape<KP>;
  constexpr int TD = S::TD, GT = S::GT, G = S::G, TC = S::TC, EPT = S::EPT;
  __shared__ double smem[S::SMEM];
  const int t = threadIdx.x, g = t / GT, gt = t % GT;
  const int ti = gt % TD, tj = gt / TD;
  const bool act = gt < TD * TD;
  const int b0 = blockIdx.x * cols, b1 = min(N, b0 + cols);
  const int per = (cols + G - 1) / G;
  const int c0 = min(b1, b0 + g * per), c1 = min(b1, c0 + per);
  const int ntiles = (per + TC - 1) / TC;
  double* tile = smem + (size_t)g * 2 * TC * KP;
  double reg[EPT];
  auto load = [&](int tt) {
#pragma unroll
    for (int e = 0; e < EPT; e++) {
      const int f = gt + e * GT, c = f / KP, i = f % KP;
      const int col = c0 + tt * TC + c;
      double x = 0.0;
      if (col < c1 && i < K) {
        x = (double)U[(size_t)col * ld + i];
        if (sub) x -= (double)sub[(size_t)col * ld + i];
      }
      reg[e] = x;
    }
  };
  double acc[4][4], sum[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    sum[r] = 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) acc[r][q] = 0.0;
  }
  load(0);
  for (int tt = 0; tt < ntiles; tt++) {
    double* tb = tile + (tt & 1) * TC * KP;
#pragma unroll
    for (int e = 0; e < EPT; e++) tb[gt + e * GT] = reg[e];
    __syncthreads();
    if (tt + 1 < ntiles) load(tt + 1);
    if (act) {
#pragma unroll 4
      for (int c = 0; c < TC; c++) {
        const double* x = tb + c * KP;
        double xi[4], xj[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          xi[r] = x[4 * ti + r];
          xj[r] = x[4 * tj + r];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          sum[r] += xi[r];
#pragma unroll
          for (int q = 0; q < 4; q++) acc[r][q] += xi[r] * xj[q];
        }
      }
    }
  }
  const int KK = K * K;
  double* out = partial + (size_t)blockIdx.x * (K + KK);
  if (G == 1) {
    if (!act) return;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 4 * ti + r;
      if (i >= K) continue;
      if (tj == 0) out[i] = sum[r];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int j = 4 * tj + q;
        if (j < K) out[K + i + j * K] = acc[r][q];
      }
    }
    return;
  }
  __syncthreads();  // tiles are dead: reuse the LDS for the group sums
  double* red = smem + (size_t)g * (K + KK);
  if (act) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 4 * ti + r;
      if (i >= K) continue;
      if (tj == 0) red[i] = sum[r];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int j = 4 * tj + q;
        if (j < K) red[K + i + j * K] = acc[r][q];
      }
    }
  }
  __syncthreads();
  for (int q = t; q < K + KK; q += S::THREADS) {
    double v = 0.0;
#pragma unroll
    for (int h = 0; h < G; h++) v += smem[(size_t)h * (K + KK) + q];
    out[q] = v;
  }
}

// The random numbers of the Normal-Wishart draw: the Bartlett factor C (upper;
// C_ii = sqrt(chi2(nu_c - i)), C_ij ~ N(0,1) for i < j: WishartUnit,
// mvnormal.cpp:217-241) at out[j K + i], and the normals of mu at out[K K + j].
// Item q: normals C[c][4b .. 4b+3] of one Philox block, then the diagonal,
// then mu's blocks.
__device__ __forceinline__ void bartlett_item(const BartlettArgs& a, int q) {
  const int K = a.K, nb = (K + 3) / 4;
  const uint32_t it = (uint32_t)(a.iter ? *a.iter : a.iter_value);
  if (q < K * nb) {
    const int c = q % K, b = q / K;
    if (4 * b + 3 <= c) return;
    double z[4];
    normal_f64x4(a.seed, (uint32_t)c, (uint32_t)b, it, make_tag(TAG_WISHART_Z, a.mode), z);
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = 4 * b + u;
      if (j > c && j < K) a.out[j * K + c] = z[u];
    }
  } else if (q < K * nb + K) {
    const int i = q - K * nb;
    a.out[i * K + i] = sqrt(2.0 * gamma_f64(a.seed, 0.5 * (a.nu_c - i), (uint32_t)i, it,
                                            make_tag(TAG_WISHART_CHI, a.mode)));
  } else if (q < K * nb + K + nb) {
    const int b = q - K * nb - K;
    double z[4];
    normal_f64x4(a.seed, 0u, (uint32_t)b, it, make_tag(TAG_NW_MU, a.mode), z);
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (4 * b + u < K) a.out[K * K + 4 * b + u] = z[u];
  }
}

// partial[0][q] = sum_b partial[b][q] in a fixed order: 16 interleaved
// strands of blocks (strand g takes b = g, g + 16, ..., eight loads in
// flight), combined in strand order.  A work-group owns 16 entries q, so
// each load instruction reads 16 consecutive entries of 4 blocks.  The first
// nbart work-groups make the draw's random numbers instead.
constexpr int kRedStrands = 16, kRedEntries = 256 / kRedStrands;

__global__ void __launch_bounds__(256) k_stats_reduce(double* partial, int nblk, int width, int nbart,
                                                      BartlettArgs bart) {
  __shared__ double red[kRedStrands][kRedEntries];
  if ((int)blockIdx.x < nbart) {
    bartlett_item(bart, blockIdx.x * 256 + threadIdx.x);
    return;
  }
  const int e = threadIdx.x % kRedEntries, g = threadIdx.x / kRedEntries;
  const int q = (blockIdx.x - nbart) * kRedEntries + e;
  double s = 0.0;
  if (q < width) {
    int b = g;
    for (; b + 7 * kRedStrands < nblk; b += 8 * kRedStrands) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = partial[(size_t)(b + kRedStrands * u) * width + q];
#pragma unroll
      for (int u = 0; u < 8; u++) s += v[u];
    }
    for (; b < nblk; b += kRedStrands) s += partial[(size_t)b * width + q];
  }
  red[g][e] = s;
  __syncthreads();
  if (g == 0 && q < width) {
    double t = red[0][e];
#pragma unroll
    for (int h = 1; h < kRedStrands; h++) t += red[h][e];
    partial[q] = t;
  }
}

static void launch_reduce(double* partial, int nblk, int width, const BartlettArgs& bart, hipStream_t s) {
  const int nred = nblk > 1 ? (width + kRedEntries - 1) / kRedEntries : 0;
  const int nb = (bart.K + 3) / 4;
  const int nbart = bart.out ? (bart.K * nb + bart.K + nb + 255) / 256 : 0;
  if (nred + nbart)
    hipLaunchKernelGGL(k_stats_reduce, dim3(nred + nbart), dim3(256), 0, s, partial, nblk, width, nbart, bart);
}

void launch_partial_reduce(double* partial, int nblk, int width, hipStream_t s) {
  launch_reduce(partial, nblk, width, BartlettArgs(), s);
}

template <typename T>
static void launch_stats(const T* U, const float* sub, int ld, int N, int K, double* partial, int nblk,
                         hipStream_t s, const BartlettArgs& bart) {
  const int KP = pad_latent(K);
  const int cols = (N + nblk - 1) / nblk;
  switch (KP) {
#define MGPU_STATS_CASE(P)                                                                                   \
  case P:                                                                                                    \
    hipLaunchKernelGGL((k_hyper_stats<T, P>), dim3(nblk), dim3(StatShape<P>::THREADS), 0, s, U, sub, ld, N, K, \
                       cols, partial);                                                                       \
    break;
    MGPU_STATS_CASE(8)
    MGPU_STATS_CASE(16)
    MGPU_STATS_CASE(32)
    MGPU_STATS_CASE(64)
    MGPU_STATS_CASE(128)
#undef MGPU_STATS_CASE
    default: break;
  }
  launch_reduce(partial, nblk, K + K * K, bart, s);
}

void launch_hyper_stats_f32(const float* U, const float* sub, int ld, int N, int K, double* partial, int nblk,
                            hipStream_t s, const BartlettArgs& bart) {
  launch_stats<float>(U, sub, ld, N, K, partial, nblk, s, bart);
}
void launch_hyper_stats_f64(const double* U, int ld, int N, int K, double* partial, int nblk, hipStream_t s,
                            const BartlettArgs& bart) {
  launch_stats<double>(U, nullptr, ld, N, K, partial, nblk, s, bart);
}

// ------------------------------------------------------------------
// Adaptive noise: SSE over the training cells (noisemodels.cpp:55-124)
// ------------------------------------------------------------------
constexpr int kNoiseThreads = 256;

int noise_sse_blocks(int N0) {
  int b = (N0 + 3) / 4;
  if (b < 1) b = 1;
  if (b > 1024) b = 1024;
  return b;
}

template <int KP>
__global__ void __launch_bounds__(kNoiseThreads) k_noise_sse(NoiseArgs a) {
  __shared__ float us[kNoiseThreads / 64][KP];
  __shared__ double red[kNoiseThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nw = gridDim.x * (kNoiseThreads / 64);
  const int no = a.nmodes - 1;
  double acc = 0.0;
  for (int row = blockIdx.x * (kNoiseThreads / 64) + w; row < a.rows0.N; row += nw) {
    for (int i = lane; i < KP; i += 64) us[w][i] = a.U0[(size_t)row * KP + i];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int beg = a.rows0.row_ptr[row], end = a.rows0.row_ptr[row + 1];
    for (int e = beg + lane; e < end; e += 64) {
      float dot = 0.f;
      const int* ix = a.rows0.idx + (size_t)e * no;
      for (int d = 0; d < a.K; d++) {
        float v = us[w][d];
        for (int m = 0; m < no; m++) v *= a.others.f[m][(size_t)ix[m] * KP + d];
        dot += v;
      }
      const double r = (double)dot - (double)a.rows0.r[e];
      acc += r * r;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if (lane == 0) red[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int q = 0; q < kNoiseThreads / 64; q++) s += red[q];
    a.partial[blockIdx.x] = s;
  }
}

void launch_noise_sse(const NoiseArgs& a, hipStream_t s) {
  switch (a.KP) {
    case 8: hipLaunchKernelGGL((k_noise_sse<8>), dim3(a.nblk), dim3(kNoiseThreads), 0, s, a); break;
    case 16: hipLaunchKernelGGL((k_noise_sse<16>), dim3(a.nblk), dim3(kNoiseThreads), 0, s, a); break;
    case 32: hipLaunchKernelGGL((k_noise_sse<32>), dim3(a.nblk), dim3(kNoiseThreads), 0, s, a); break;
    case 64: hipLaunchKernelGGL((k_noise_sse<64>), dim3(a.nblk), dim3(kNoiseThreads), 0, s, a); break;
    default: hipLaunchKernelGGL((k_noise_sse<128>), dim3(a.nblk), dim3(kNoiseThreads), 0, s, a); break;
  }
}

// alpha ~ Gamma(a0 + nnz/2, 1/(b0 + SSE/2)), clamped to alpha_max
__global__ void k_noise_draw(NoiseDrawArgs a) {
  __shared__ double red[256];
  double s = 0.0;
  for (int b = threadIdx.x; b < a.nblk; b += 256) s += a.partial[b];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double sse = red[0];
    const double aN = 0.5 + a.nnz / 2.0;
    const double bN = a.b0 + sse / 2.0;
    double al = gamma_f64(a.seed, aN, 0u, (uint32_t)*a.iter, make_tag(TAG_NOISE, 0)) / bN;
    if (al > a.alpha_max) al = a.alpha_max;
    *a.alpha = al;
    if (a.sse_out) *a.sse_out = sse;
  }
}

void launch_noise_draw(const NoiseDrawArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_noise_draw, dim3(1), dim3(256), 0, s, a);
}

// ------------------------------------------------------------------
// Evaluation: eval_rmse / eval_rmse_tensor (bpmfutils.h:86-114,
// bpmfutils.cpp:10-73) with Welford running mean and variance.
// A group of KP/4 lanes handles one test cell: each lane multiplies one
// float4 of the factor columns, the group sums by shuffles, and the group's
// first lane updates the FP64 running mean/variance and squared errors.
// ------------------------------------------------------------------
constexpr int kEvalThreads = 256;
int eval_blocks(int ntest) {
  int b = (ntest + kEvalThreads * 2 - 1) / (kEvalThreads * 2);
  if (b < 1) b = 1;
  if (b > 2048) b = 2048;
  return b;
}

template <int KP, int NM, bool PROBIT>
__global__ void __launch_bounds__(kEvalThreads) k_eval(EvalArgs a) {
  constexpr int G = KP / 4;  // lanes per test cell
  __shared__ double red[2][kEvalThreads / 64];
  const int it = *a.iter;
  const int n = it < a.burnin ? 0 : it - a.burnin;
  const int sub = threadIdx.x % G;
  const int cells_per_block = kEvalThreads / G;
  // U consecutive cells per lane group and loop step: their index loads,
  // then their factor-row loads, are issued together, and after the
  // lane-group sums lane u of the group finishes cell u, so the FP64 running
  // mean and variance run once per U cells instead of once per cell
  // (U <= G: every cell needs an owner lane in its group)
  constexpr int U = G < 4 ? G : 4;
  double se = 0.0, se_avg = 0.0;
  // NM modes (NM = kMaxOther + 1: nm = the run-time count, at most NM)
  const int nm = NM <= kMaxOther ? NM : a.nmodes;
  for (int q0 = blockIdx.x * cells_per_block * U; q0 < a.ntest; q0 += gridDim.x * cells_per_block * U) {
    int qs[U], ix[U][NM];
#pragma unroll
    for (int u = 0; u < U; u++) {
      qs[u] = q0 + (threadIdx.x / G) * U + u;
#pragma unroll
      for (int m = 0; m < NM; m++) ix[u][m] = (qs[u] < a.ntest && m < nm) ? a.idx[(size_t)qs[u] * nm + m] : -1;
    }
    float dot[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      dot[u] = 0.f;
      if (ix[u][0] >= 0) {
        float4 v = reinterpret_cast<const float4*>(a.f[0] + (size_t)ix[u][0] * KP)[sub];
#pragma unroll
        for (int m = 1; m < NM; m++) {
          if (m >= nm) break;
          const float4 w = reinterpret_cast<const float4*>(a.f[m] + (size_t)ix[u][m] * KP)[sub];
          v.x *= w.x;
          v.y *= w.y;
          v.z *= w.z;
          v.w *= w.w;
        }
        dot[u] = (v.x + v.y) + (v.z + v.w);
      }
    }
    float d = 0.f;
    int q = a.ntest;
#pragma unroll
    for (int u = 0; u < U; u++) {
      float du = dot[u];
#pragma unroll
      for (int off = 1; off < G; off <<= 1) du += __shfl_xor(du, off, G);
      if (sub == u) {
        d = du;
        q = qs[u];
      }
    }
    if (sub < U && q < a.ntest) {
      double p;
      if constexpr (PROBIT) {
        p = 0.5 * erfc(-(double)d * M_SQRT1_2);
        a.pred1[q] = p;
      } else {
        p = a.mean + (double)d;
      }
      double pa;
      if (n == 0) {
        pa = p;
        a.pred_var[q] = 0.0;
      } else {
        const double delta = p - a.pred[q];
        pa = a.pred[q] + delta / (n + 1);
        a.pred_var[q] += delta * (p - pa);
      }
      a.pred[q] = pa;
      const double y = a.vals[q];
      se += (y - p) * (y - p);
      se_avg += (y - pa) * (y - pa);
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    se += __shfl_down(se, off, 64);
    se_avg += __shfl_down(se_avg, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = se;
    red[1][threadIdx.x >> 6] = se_avg;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s0 = 0.0, s1 = 0.0;
    for (int w = 0; w < kEvalThreads / 64; w++) {
      s0 += red[0][w];
      s1 += red[1][w];
    }
    a.partial[2 * blockIdx.x] = s0;
    a.partial[2 * blockIdx.x + 1] = s1;
  }
}

__global__ void __launch_bounds__(256) k_eval_finish(EvalArgs a) {
  __shared__ double red[2][256];
  double s0 = 0.0, s1 = 0.0;
  for (int b = threadIdx.x; b < a.nblk; b += 256) {
    s0 += a.partial[2 * b];
    s1 += a.partial[2 * b + 1];
  }
  red[0][threadIdx.x] = s0;
  red[1][threadIdx.x] = s1;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      red[0][threadIdx.x] += red[0][threadIdx.x + off];
      red[1][threadIdx.x] += red[1][threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    // an empty test set gives sqrt(0 / 0) = NaN (bpmfutils.h:110-112)
    a.out[0] = a.ntest == 0 ? NAN : sqrt(red[0][0] / (double)a.ntest);
    a.out[1] = a.ntest == 0 ? NAN : sqrt(red[1][0] / (double)a.ntest);
  }
}

template <int KP>
static void launch_eval_k(const EvalArgs& a, hipStream_t s) {
  if (a.probit) {  // matrix data only (ProbitNoise::evalModel(TensorData) throws)
    hipLaunchKernelGGL((k_eval<KP, 2, true>), dim3(a.nblk), dim3(kEvalThreads), 0, s, a);
    return;
  }
  switch (a.nmodes) {
    case 2: hipLaunchKernelGGL((k_eval<KP, 2, false>), dim3(a.nblk), dim3(kEvalThreads), 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_eval<KP, 3, false>), dim3(a.nblk), dim3(kEvalThreads), 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_eval<KP, 4, false>), dim3(a.nblk), dim3(kEvalThreads), 0, s, a); break;
    case 5: hipLaunchKernelGGL((k_eval<KP, 5, false>), dim3(a.nblk), dim3(kEvalThreads), 0, s, a); break;
    default: hipLaunchKernelGGL((k_eval<KP, kMaxOther + 1, false>), dim3(a.nblk), dim3(kEvalThreads), 0, s, a); break;
  }
}

void launch_eval(const EvalArgs& a, hipStream_t s) {
  if (a.ntest > 0) {
    switch (a.KP) {
      case 8: launch_eval_k<8>(a, s); break;
      case 16: launch_eval_k<16>(a, s); break;
      case 32: launch_eval_k<32>(a, s); break;
      case 64: launch_eval_k<64>(a, s); break;
      default: launch_eval_k<128>(a, s); break;
    }
  }
  hipLaunchKernelGGL(k_eval_finish, dim3(1), dim3(256), 0, s, a);
}

__global__ void k_advance_iter(int* iter) {
  if (threadIdx.x == 0) *iter += 1;
}
void launch_advance_iter(int* iter, hipStream_t s) { hipLaunchKernelGGL(k_advance_iter, dim3(1), dim3(64), 0, s, iter); }

// ------------------------------------------------------------------
// RNG probes used by the parity tests
// ------------------------------------------------------------------
__global__ void k_rng_probe(uint64_t seed, uint32_t c0, uint32_t it, uint32_t tag, int n, uint32_t* bits,
                            float* z32, double* z64) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  if ((j & 3) == 0) {
    uint32_t w[4];
    philox_at(seed, c0, (uint32_t)(j >> 2), it, tag, w);
    for (int q = 0; q < 4 && j + q < n; q++) bits[j + q] = w[q];
  }
  z32[j] = normal_f32(seed, c0, (uint32_t)j, it, tag);
  z64[j] = normal_f64(seed, c0, (uint32_t)j, it, tag);
}
void launch_rng_probe(uint64_t seed, uint32_t c0, uint32_t it, uint32_t tag, int n, uint32_t* bits, float* z32,
                      double* z64, hipStream_t s) {
  hipLaunchKernelGGL(k_rng_probe, dim3((n + 255) / 256), dim3(256), 0, s, seed, c0, it, tag, n, bits, z32, z64);
}

__global__ void k_gamma_probe(uint64_t seed, const double* shapes, int n, uint32_t it, uint32_t tag, double* out) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) out[j] = gamma_f64(seed, shapes[j], (uint32_t)j, it, tag);
}
void launch_gamma_probe(uint64_t seed, const double* shapes, int n, uint32_t it, uint32_t tag, double* out,
                        hipStream_t s) {
  hipLaunchKernelGGL(k_gamma_probe, dim3((n + 255) / 256), dim3(256), 0, s, seed, shapes, n, it, tag, out);
}

}  // namespace mgpu
