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
// in FP64 and reduced in a fixed order, beside work-groups
// that make the draw's random numbers (which need no statistics); the K x K
// draw then runs in one work-group (nwdraw.hip).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace mgpu {

// ------------------------------------------------------------------
// Sufficient statistics of x_n = U[:, n] - sub[:, n] (sub optional, FP32, same
// ld) in FP64: sum_n x_n and sum_n x_n x_n^T.
//
// The scatter is a product with the columns as reduction index, so it runs on
// v_mfma_f64_16x16x4f64, four columns a step: lane l holds entry l % 16 of each
// 16-component tile of column l / 16, which is the A and the B operand of every
// tile product at once.  No LDS between the loads and the products; only lower
// tiles are formed.  With KP <= 64 each wave takes its own columns and holds
// every tile (10 at most), and a work-group's four waves are summed through
// LDS at the end; above, the 36 tiles are shared by the waves (rows w and 7 - w
// of the triangle on wave w: nine each), which walk the same columns.
// FP32 factors have their components dealt to the tiles in turn (component
// c NT + t is entry c of tile t), so a lane's NT values are one contiguous load.
// Statistics and reduction before (4 x 4 register tiles per thread over LDS
// tiles of 16 columns, partials of the whole K x K) and now, alone on the card:
// 100003 x 64 FP64 140 -> 24 us (51 MB: 2.6 TB/s in the first kernel), 3001 x
// 128 FP32 37 -> 15 us; with the draw, 138000 x 32 FP32 79 -> 35 us.
// ------------------------------------------------------------------
typedef double f64x4 __attribute__((ext_vector_type(4)));

static int stats_tiles(int K) { return K <= 16 ? 1 : K <= 32 ? 2 : K <= 64 ? 4 : 8; }
// doubles of a block's partial: the tiles' sums, then the lower tiles
static int stats_width(int K) {
  const int nt = stats_tiles(K);
  return 16 * nt + 128 * nt * (nt + 1);
}
// One work-group per 32 columns up to one per CU.  Above K = 64 a wave has one
// step's loads in flight, so many columns take two work-groups a CU; fewer do not,
// because a partial is 74 KB and the reduction's reads count.  Statistics and draw
// in us with 128 | 256 | 512 | 1024 work-groups, K = 128, FP32:
//   10000 columns   77 | 72 | 74 | 73      100000    232 | 147 | 123 | 129
//   20000           94 | 79 | 77 | 81     1000000   1789 | 942 | 684 | 661
int hyper_stats_blocks(int N, int K) {
  const int cap = K > 64 && N >= 32768 ? 512 : 256;
  return std::max(1, std::min(cap, (N + 31) / 32));
}
size_t hyper_stats_doubles(int nblk, int K) { return (size_t)2 * (K + K * K) + (size_t)nblk * stats_width(K); }

// component of entry c of tile t
template <typename T, int NT>
__host__ __device__ __forceinline__ constexpr int stats_component(int t, int c) {
  return sizeof(T) == 4 ? c * NT + t : 16 * t + c;
}

template <typename T, int NT>
__global__ void __launch_bounds__(256)
    k_hyper_stats(const T* __restrict__ U, const float* __restrict__ sub, const int* __restrict__ skip, int ld, int N,
                  int K, int cols, double* __restrict__ partial) {
  constexpr bool kShared = NT > 4;                      // the waves share the tiles
  constexpr int NTILE = NT * (NT + 1) / 2;
  constexpr int WIDTH = 16 * NT + 256 * NTILE;
  constexpr int STEP = kShared ? 4 : 16;                // columns a work-group takes per step
  constexpr int AHEAD = NT <= 2 ? 4 : NT == 4 ? 2 : 1;  // steps whose loads are in flight
  __shared__ double red[kShared ? 1 : 2 * WIDTH];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int b0 = blockIdx.x * cols, b1 = min(N, b0 + cols);
  const int first = b0 + (kShared ? 0 : 4 * wave) + g;
  f64x4 acc[kShared ? 12 : NTILE];
#pragma unroll
  for (int q = 0; q < (kShared ? 12 : NTILE); q++) acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
  double sum[NT];
#pragma unroll
  for (int q = 0; q < NT; q++) sum[q] = 0.0;

  T raw[AHEAD][NT];
  float rsub[AHEAD][NT];
  int out_of[AHEAD];  // columns left out (FP64 input only)
  auto load = [&](T(&x)[NT], float(&y)[NT], int& o, int col) {
    o = sizeof(T) == 8 && skip ? skip[min(col, N - 1)] : -1;
    const size_t at = (size_t)min(col, N - 1) * ld;
    if constexpr (sizeof(T) == 4 && NT > 1) {  // ld = 16 NT: entries c NT .. c NT + NT - 1
      typedef float vec __attribute__((ext_vector_type(NT == 2 ? 2 : 4)));
      constexpr int P = NT == 2 ? 2 : 4;
#pragma unroll
      for (int p = 0; p < NT / P; p++) {
        const vec v = *reinterpret_cast<const vec*>(U + at + c * NT + p * P);
        vec w = 0.f;
        if (sub) w = *reinterpret_cast<const vec*>(sub + at + c * NT + p * P);
#pragma unroll
        for (int q = 0; q < P; q++) {
          x[p * P + q] = v[q];
          y[p * P + q] = w[q];
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < NT; q++) {
        const int k = min(stats_component<T, NT>(q, c), ld - 1);
        x[q] = U[at + k];
        y[q] = sub ? sub[at + k] : 0.f;
      }
    }
  };
  if (b0 < b1) {
#pragma unroll
    for (int u = 0; u < AHEAD; u++) load(raw[u], rsub[u], out_of[u], first + u * STEP);
  }
  for (int n0 = first - g; n0 < b1; n0 += AHEAD * STEP) {
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      const int col = n0 + g + u * STEP;
      const bool in = col < b1 && out_of[u] < 0;
      double x[NT];
#pragma unroll
      for (int q = 0; q < NT; q++) {
        double v = (double)raw[u][q];
        if (sizeof(T) == 4) v -= (double)rsub[u][q];
        x[q] = (in && stats_component<T, NT>(q, c) < K) ? v : 0.0;
        sum[q] += x[q];
      }
      load(raw[u], rsub[u], out_of[u], col + AHEAD * STEP);
      if constexpr (!kShared) {
        int id = 0;
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
          for (int j = 0; j <= i; j++, id++)
            acc[id] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], x[j], acc[id], 0, 0, 0);
      } else {
        const double lo = wave == 0 ? x[0] : wave == 1 ? x[1] : wave == 2 ? x[2] : x[3];
        const double hi = wave == 0 ? x[7] : wave == 1 ? x[6] : wave == 2 ? x[5] : x[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (j <= wave) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(lo, x[j], acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 8; j++)
          if (j <= 7 - wave) acc[4 + j] = __builtin_amdgcn_mfma_f64_16x16x4f64(hi, x[j], acc[4 + j], 0, 0, 0);
      }
    }
  }
  // sums over the four columns of a step
#pragma unroll
  for (int q = 0; q < NT; q++) {
    sum[q] += __shfl_xor(sum[q], 16, 64);
    sum[q] += __shfl_xor(sum[q], 32, 64);
  }
  double* out = partial + (size_t)blockIdx.x * WIDTH;
  if constexpr (kShared) {
    if (wave == 0 && g == 0) {
#pragma unroll
      for (int q = 0; q < NT; q++) out[16 * q + c] = sum[q];
    }
    auto store = [&](int i, int j, const f64x4& v) {
      double* o = out + 16 * NT + 256 * (i * (i + 1) / 2 + j);
#pragma unroll
      for (int u = 0; u < 4; u++) o[64 * u + lane] = v[u];
    };
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (j <= wave) store(wave, j, acc[j]);
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (j <= 7 - wave) store(7 - wave, j, acc[4 + j]);
  } else {
    // waves 1 and 3 to LDS, added by 0 and 2; then 2 to LDS, added by 0
    auto put = [&](double* r) {
      if (g == 0) {
#pragma unroll
        for (int q = 0; q < NT; q++) r[16 * q + c] = sum[q];
      }
#pragma unroll
      for (int q = 0; q < NTILE; q++)
#pragma unroll
        for (int u = 0; u < 4; u++) r[16 * NT + 256 * q + 64 * u + lane] = acc[q][u];
    };
    auto add = [&](const double* r) {
#pragma unroll
      for (int q = 0; q < NT; q++) sum[q] += r[16 * q + c];
#pragma unroll
      for (int q = 0; q < NTILE; q++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[q][u] += r[16 * NT + 256 * q + 64 * u + lane];
    };
    if (wave & 1) put(red + (wave >> 1) * WIDTH);
    __syncthreads();
    if (!(wave & 1)) add(red + (wave >> 1) * WIDTH);
    __syncthreads();
    if (wave == 2) put(red);
    __syncthreads();
    if (wave == 0) {
      add(red);
      put(out);
    }
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

// sum_b partial[b][q] in a fixed order: 16 interleaved strands of blocks
// (strand g takes b = g, g + 16, ..., eight loads in flight), combined in
// strand order.  A work-group owns 16 entries q, so each load instruction reads
// 16 consecutive entries of 4 blocks.  Valid on threads 0 .. 15 (entry
// threadIdx.x of the work-group).
constexpr int kRedStrands = 16, kRedEntries = 256 / kRedStrands;

__device__ __forceinline__ double strands_sum(const double* partial, int nblk, int width, int q0) {
  __shared__ double red[kRedStrands][kRedEntries];
  const int e = threadIdx.x % kRedEntries, g = threadIdx.x / kRedEntries;
  const int q = q0 + e;
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
  double t = 0.0;
  if (g == 0) {
    t = red[0][e];
#pragma unroll
    for (int h = 1; h < kRedStrands; h++) t += red[h][e];
  }
  return t;
}

// partial[0][q] = sum_b partial[b][q], in place
__global__ void __launch_bounds__(256) k_partial_reduce(double* partial, int nblk, int width) {
  const int q = blockIdx.x * kRedEntries + threadIdx.x;
  const double t = strands_sum(partial, nblk, width, blockIdx.x * kRedEntries);
  if (threadIdx.x < kRedEntries && q < width) partial[q] = t;
}

void launch_partial_reduce(double* partial, int nblk, int width, hipStream_t s) {
  if (nblk > 1)
    hipLaunchKernelGGL(k_partial_reduce, dim3((width + kRedEntries - 1) / kRedEntries), dim3(256), 0, s, partial, nblk,
                       width);
}

// The statistics' partials summed into out = (sum (K), scatter (K x K)).  The
// first nbart work-groups make the Normal-Wishart draw's random numbers
// instead, which need no statistics.
template <typename T, int NT>
__global__ void __launch_bounds__(256) k_stats_reduce(const double* __restrict__ partial, int nblk, int K,
                                                      double* __restrict__ out, int nbart, BartlettArgs bart) {
  if ((int)blockIdx.x < nbart) {
    bartlett_item(bart, blockIdx.x * 256 + threadIdx.x);
    return;
  }
  constexpr int WIDTH = 16 * NT + 128 * NT * (NT + 1);
  const int q0 = (blockIdx.x - nbart) * kRedEntries, c = threadIdx.x;
  const double t = strands_sum(partial, nblk, WIDTH, q0);
  if (c >= kRedEntries) return;
  if (q0 < 16 * NT) {
    const int k = stats_component<T, NT>(q0 / 16, c);
    if (k < K) out[k] = t;
    return;
  }
  const int id = (q0 - 16 * NT) / 256, r = (q0 - 16 * NT) % 256 / 16;
  int ti = 0;
  while ((ti + 1) * (ti + 2) / 2 <= id) ti++;
  const int tj = id - ti * (ti + 1) / 2;
  const int i = stats_component<T, NT>(ti, r), j = stats_component<T, NT>(tj, c);
  if (i < K && j < K) {
    out[K + i + j * K] = t;
    if (ti != tj) out[K + j + i * K] = t;
  }
}

template <typename T>
static void launch_stats(const T* U, const float* sub, const int* skip, int ld, int N, int K, double* ws, int nblk, hipStream_t s,
                         const BartlettArgs& bart) {
  double* partial = ws + 2 * (K + K * K);
  const int cols = (N + nblk - 1) / nblk;
  const int nred = stats_width(K) / kRedEntries, nb = (bart.K + 3) / 4;
  const int nbart = bart.out ? (bart.K * nb + bart.K + nb + 255) / 256 : 0;
  switch (stats_tiles(K)) {
#define MGPU_STATS_CASE(NT)                                                                                       \
  case NT:                                                                                                        \
    hipLaunchKernelGGL((k_hyper_stats<T, NT>), dim3(nblk), dim3(256), 0, s, U, sub, skip, ld, N, K, cols,      \
                       partial);                                                                                  \
    hipLaunchKernelGGL((k_stats_reduce<T, NT>), dim3(nred + nbart), dim3(256), 0, s, partial, nblk, K, ws, nbart, \
                       bart);                                                                                     \
    break;
    MGPU_STATS_CASE(1)
    MGPU_STATS_CASE(2)
    MGPU_STATS_CASE(4)
    MGPU_STATS_CASE(8)
#undef MGPU_STATS_CASE
    default: break;
  }
}

void launch_hyper_stats_f32(const float* U, const float* sub, int ld, int N, int K, double* ws, int nblk,
                            hipStream_t s, const BartlettArgs& bart) {
  launch_stats<float>(U, sub, nullptr, ld, N, K, ws, nblk, s, bart);
}
void launch_hyper_stats_f64(const double* U, int ld, int N, int K, double* ws, int nblk, hipStream_t s,
                            const BartlettArgs& bart, const int* skip) {
  launch_stats<double>(U, nullptr, skip, ld, N, K, ws, nblk, s, bart);
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
