// nwdraw.hip -- the Normal-Wishart draw of one mode (CondNormalWishart,
// mvnormal.cpp:314-336), FP64, K <= 128.
//
// With X = T + S + kappa mu0 mu0^T - kappa_c mu_c mu_c^T the Bartlett draw is
//   Lambda = L_T (C^T C) L_T^T,  L_T = chol(X^{-1})
// (Wishart, mvnormal.cpp:243-266; C upper, WishartUnit, mvnormal.cpp:217-241).
// X = U U^T with U upper triangular (Cholesky from the last row up) gives
// L_T = U^{-T} (the lower Cholesky factor is unique), so Lambda = B B^T with
// B = U^{-T} C^T: one factorisation and one triangular solve.  B is lower
// triangular with a positive diagonal, i.e. chol(Lambda), hence
// mu = mu_c + B^{-T} z / sqrt(kappa_c) (MvNormal_prec, mvnormal.cpp:169-184)
// and Lambda mu = B (B^T mu_c + z / sqrt(kappa_c)).
//
// One work-group per draw, everything in 16 x 16 FP64 tiles
// (v_mfma_f64_16x16x4f64).  The draw sits on the sampler's critical path and
// is bound by latency, not by work: a chain of K pivots.  Tiles cut what used
// to be a barrier (or an LDS round trip) per column or four columns to two
// barriers per 16: the pivots of a diagonal tile run in one wave's registers
// (which also leave U_kk^{-1}, so panels and solves are products), the
// trailing update of the other tiles runs beside the next diagonal tile, and
// the triangular solve needs no barrier at all: a wave owns whole block
// columns of B, and the accumulator layout of a product is the operand layout
// of the next.  Random draws are made beforehand by the work-groups of
// launch_hyper_stats' reduction, side by side.
// Per draw, launched alone, before (one wave's column-by-column chain at
// K <= 64, packed triangles with two barriers per four columns above) and now:
// see the table at launch_nw_draw.
#include <atomic>

#include "common.h"
#include "model.h"

namespace mgpu {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// A 16 x 16 tile in LDS: row r at 16 r, its columns XORed with r, so that both
// ways the matrix unit's operands are read (64 consecutive entries; 16 rows of
// 4 columns) touch every bank once.
__device__ __forceinline__ int tix(int r, int c) { return 16 * r + (c ^ r); }
// tile (i, j), j <= i, of a packed lower triangle of tiles
__device__ __forceinline__ int ltile(int i, int j) { return 256 * (i * (i + 1) / 2 + j); }

// 1/sqrt(d), d > 0: the hardware estimate (v_rsq_f64) refined by two
// Newton-Raphson steps for f(y) = y^-2 - d, y <- y (3 - d y^2) / 2, each of
// which roughly squares the relative error
__device__ __forceinline__ double rsqrt_nr(double d) {
  double y = __builtin_amdgcn_rsq(d);
  const double h = 0.5 * d;
  y = y * fma(-h * y, y, 1.5);
  y = y * fma(-h * y, y, 1.5);
  return y;
}

// Operands of D = A B, lane l, step s of 4: A[l % 16][4s + l / 16],
// B[4s + l / 16][l % 16]; D[4v + l / 16][l % 16] in register v.  `rows` reads
// M[4s + l / 16][l % 16] (M as B operand, or M^T as A operand), `cols` reads
// M[l % 16][4s + l / 16] (M as A operand, or M^T as B operand).
__device__ __forceinline__ f64x4 rows(const double* M, int lane) {
  f64x4 v;
#pragma unroll
  for (int s = 0; s < 4; s++) v[s] = M[tix(4 * s + (lane >> 4), lane & 15)];
  return v;
}
__device__ __forceinline__ f64x4 cols(const double* M, int lane) {
  f64x4 v;
#pragma unroll
  for (int s = 0; s < 4; s++) v[s] = M[tix(lane & 15, 4 * s + (lane >> 4))];
  return v;
}
__device__ __forceinline__ void put(double* M, int lane, f64x4 v) {
#pragma unroll
  for (int s = 0; s < 4; s++) M[tix(4 * s + (lane >> 4), lane & 15)] = v[s];
}
__device__ __forceinline__ f64x4 mul_add(f64x4 a, f64x4 b, f64x4 c) {
#pragma unroll
  for (int s = 0; s < 4; s++) c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], c, 0, 0, 0);
  return c;
}

// One wave: the diagonal tile X = U U^T, replaced by U^{-1}.  Lanes 0-15 hold
// the columns of X, lanes 16-31 those of the identity; the row operations that
// take X to U^T (pivots from the last row up) take the identity to U^{-1}.
// Returns true if a pivot was not positive (it is replaced by 1).
__device__ __forceinline__ bool diag_factor(double* X, int lane) {
  double a[16];
  const int c = lane & 15;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const double x = X[tix(r, c)];
    a[r] = lane < 16 ? x : (lane == 16 + r ? 1.0 : 0.0);
  }
  bool bad = false;
#pragma unroll
  for (int p = 15; p >= 0; p--) {
    const double d = rdlane(a[p], p);
    const bool b = !(d > 0.0);
    bad = bad || b;
    a[p] *= rsqrt_nr(b ? 1.0 : d);
#pragma unroll
    for (int i = p - 1; i >= 0; i--) a[i] = fma(-rdlane(a[p], i), a[p], a[i]);
  }
  if (lane >= 16 && lane < 32) {
#pragma unroll
    for (int r = 0; r < 16; r++) X[tix(r, c)] = a[r];
  }
  return bad;
}

// NTM bounds the tiles per dimension, W is the number of waves.
template <int NTM, int W>
__global__ void __launch_bounds__(64 * W) k_nw_draw(NWArgs a) {
  extern __shared__ double sm[];
  const int K = a.K, KK = K * K, nt = (K + 15) / 16, ntile = nt * (nt + 1) / 2;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane >> 4, lc = lane & 15;
  double* X = sm;                 // X, then U^T (lower tiles; U_kk^{-1} on the diagonal), then B
  double* v_mu = X + 256 * ntile;  // mu_c
  double* v_z = v_mu + 16 * nt;   // z / sqrt(kappa_c)
  double* v_w = v_z + 16 * nt;    // B^T mu_c + z / sqrt(kappa_c)
  const double kappa_c = a.kappa + a.N;
  const double* S = a.partial + K;
  bool bad = false;

  // 1. the wave's block column of C^T, on its way while X is factored.  Wave
  //    w takes column w and wave 4 + w column nt - 1 - w, so that the long
  //    and the short columns share a SIMD
  int j = wave < 4 ? wave : nt - 1 - (wave - 4);
  if (wave < 4 ? j >= nt : j < 4) j = nt;  // no column
  f64x4 T[NTM];
#pragma unroll
  for (int q = 0; q < NTM; q++)
    if (j + q < nt) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * (j + q) + 4 * v + lr, c = 16 * j + lc;
        const double x = a.bart[(r < K && c < K) ? r * K + c : 0];
        T[q][v] = (r < K && c <= r) ? x : (r >= K && r == c ? 1.0 : 0.0);
      }
    }

  // 2. X (mvnormal.cpp:322-325; Macau adds lambda_beta beta beta^T to T,
  //    latentprior.cpp:258-260), lower tiles, the entries of T's and S's upper
  //    triangles; the identity beyond K
  const double lb = a.BBt_partial ? *a.lambda_beta : 0.0;
  const double* bbt = a.BBt_partial ? a.BBt_partial + K : S;
  constexpr int PER = (NTM * (NTM + 1) / 2 + W - 1) / W;
  f64x4 x[PER];
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int id = wave + q * W;
    if (id < ntile) {
      int ti = 0;
      while ((ti + 1) * (ti + 2) / 2 <= id) ti++;
      const int tj = id - ti * (ti + 1) / 2;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * ti + 4 * v + lr, c = 16 * tj + lc;
        const int lo = min(min(r, c), K - 1), hi = min(max(r, c), K - 1), e = lo + hi * K;
        x[q][v] = a.WI[e] + lb * bbt[e] + S[e] + a.kappa * a.mu0[lo] * a.mu0[hi];
      }
    }
  }
  for (int k = t; k < 16 * nt; k += 64 * W) {
    const bool in = k < K;
    v_mu[k] = in ? (a.kappa * a.mu0[k] + a.partial[k]) / kappa_c : 0.0;
    v_z[k] = in ? a.bart[KK + k] / sqrt(kappa_c) : 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int id = wave + q * W;
    if (id < ntile) {
      int ti = 0;
      while ((ti + 1) * (ti + 2) / 2 <= id) ti++;
      const int tj = id - ti * (ti + 1) / 2;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * ti + 4 * v + lr, c = 16 * tj + lc;
        const double y = x[q][v] - kappa_c * v_mu[r] * v_mu[c];
        x[q][v] = (r < K && c < K) ? y : (r == c ? 1.0 : 0.0);
      }
      put(X + 256 * id, lane, x[q]);
    }
  }
  __syncthreads();

  // 3. X = U U^T, block columns from the last; tile (k, i) below the diagonal
  //    becomes U_ik^T
  if (wave == 0) bad = diag_factor(X + ltile(nt - 1, nt - 1), lane);
  for (int k = nt - 1; k > 0; k--) {
    __syncthreads();
    for (int i = wave; i < k; i += W) {  // U_ik^T = U_kk^{-1} X_ki
      double* P = X + ltile(k, i);
      put(P, lane, mul_add(cols(X + ltile(k, k), lane), rows(P, lane), f64x4{0.0, 0.0, 0.0, 0.0}));
    }
    __syncthreads();
    // X_im -= U_ik U_mk^T: wave 0 takes the next diagonal tile and factors
    // it, the others share the rest
    for (int id = wave == 0 ? ltile(k - 1, k - 1) / 256 : wave - 1; id < k * (k + 1) / 2; id += W - 1) {
      int i = 0;
      while ((i + 1) * (i + 2) / 2 <= id) i++;
      const int m = id - i * (i + 1) / 2;
      if (wave != 0 && i == k - 1 && m == k - 1) continue;
      double* P = X + ltile(i, m);
      const f64x4 u = rows(X + ltile(k, i), lane);
      put(P, lane, mul_add(-u, rows(X + ltile(k, m), lane), rows(P, lane)));
      if (wave == 0) break;
    }
    if (wave == 0) {
      lds_wait();
      bad = diag_factor(X + ltile(k - 1, k - 1), lane) || bad;
    }
  }
  __syncthreads();

  // 4. U^T B = C^T, forward, one block column per wave
#pragma unroll
  for (int q = 0; q < NTM; q++)
    if (j + q < nt) {
      T[q] = mul_add(rows(X + ltile(j + q, j + q), lane), T[q], f64x4{0.0, 0.0, 0.0, 0.0});
#pragma unroll
      for (int p = q + 1; p < NTM; p++)
        if (j + p < nt) T[p] = mul_add(-cols(X + ltile(j + p, j + q), lane), T[q], T[p]);
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NTM; q++)
    if (j + q < nt) put(X + ltile(j + q, j), lane, T[q]);
  __syncthreads();

  if (wave == 0) {
    // 5. mu: B^T x = z / sqrt(kappa_c) from the last row up, lane l holding
    //    x_l and x_{l+64}
    double y[2], inv[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int i = lane + 64 * h, ti = min(i >> 4, nt - 1);
      y[h] = i < 16 * nt ? v_z[i] : 0.0;
      inv[h] = 1.0 / X[ltile(ti, ti) + tix(i & 15, i & 15)];
    }
    for (int ti = nt - 1; ti >= 0; ti--) {  // 16 rows: their entries of B first, then the chain
      const bool upper = NTM > 4 && ti >= 4;
      double b[16][2];
#pragma unroll
      for (int r = 0; r < 16; r++)
#pragma unroll
        for (int h = 0; h < (NTM > 4 ? 2 : 1); h++) {
          const int i = lane + 64 * h;
          const double v = X[ltile(ti, min(i >> 4, ti)) + tix(r, i & 15)];
          b[r][h] = i < 16 * ti + r ? v : 0.0;
        }
#pragma unroll
      for (int r = 15; r >= 0; r--) {
        const double xr = rdlane(upper ? y[1] * inv[1] : y[0] * inv[0], (16 * ti + r) & 63);
#pragma unroll
        for (int h = 0; h < (NTM > 4 ? 2 : 1); h++) y[h] = fma(-b[r][h], xr, y[h]);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int i = lane + 64 * h;
      if (i < K) a.mu[i] = v_mu[i] + y[h] * inv[h];
    }
  } else if (wave == 1) {
    // 6. Lambda mu = B (B^T mu_c + z / sqrt(kappa_c))
    for (int c = lane; c < 16 * nt; c += 64) {
      double s[4] = {v_z[c], 0.0, 0.0, 0.0};
      for (int r = c & ~15; r < K; r += 4)
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] += X[ltile(r >> 4, c >> 4) + tix((r + u) & 15, c & 15)] * v_mu[r + u];
      v_w[c] = (s[0] + s[1]) + (s[2] + s[3]);
    }
    lds_wait();
    for (int r = lane; r < a.KP; r += 64) {
      double s[4] = {0.0, 0.0, 0.0, 0.0};
      if (r < K)
        for (int c = 0; c <= (r | 15); c += 4)
#pragma unroll
          for (int u = 0; u < 4; u++) s[u] += X[ltile(r >> 4, c >> 4) + tix(r & 15, (c + u) & 15)] * v_w[c + u];
      a.Lmu_f[r] = (float)((s[0] + s[1]) + (s[2] + s[3]));
    }
  } else {
    // 7. Lambda = B B^T, longest tiles first
    int id = 0;
    for (int tj = nt - 1; tj >= 0; tj--)
      for (int ti = tj; ti < nt; ti++, id++) {
        if (id % (W - 2) != wave - 2) continue;
        f64x4 d = {0.0, 0.0, 0.0, 0.0};
        for (int k = 0; k <= tj; k++) d = mul_add(cols(X + ltile(ti, k), lane), cols(X + ltile(tj, k), lane), d);
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r = 16 * ti + 4 * v + lr, c = 16 * tj + lc;
          if (r < K && c < K) {
            a.Lambda[c + r * K] = d[v];
            a.Lambda_f[c + r * a.KP] = (float)d[v];
            if (ti != tj) {
              a.Lambda[r + c * K] = d[v];
              a.Lambda_f[r + c * a.KP] = (float)d[v];
            }
          }
        }
      }
  }
  // 8. the FP32 copy is the identity beyond K; chol(Lambda) = B
  if (a.KP > K)
    for (int e = t; e < a.KP * a.KP; e += 64 * W) {
      const int r = e % a.KP, c = e / a.KP;
      if (r >= K || c >= K) a.Lambda_f[e] = r == c ? 1.f : 0.f;
    }
  if (a.Lchol)
    for (int e = t; e < KK; e += 64 * W) {
      const int r = e % K, c = e / K;
      a.Lchol[e] = r >= c ? X[ltile(r >> 4, min(c >> 4, r >> 4)) + tix(r & 15, c & 15)] : 0.0;
    }
  if (t == 0) {
    if (bad && a.fail) atomicMax(a.fail, kFailNormalWishart);
    if (a.status) *a.status = bad ? kFailNormalWishart : 0;
  }
}

template <int NTM, int W>
void launch(const NWArgs& a, hipStream_t s) {
  const int nt = (a.K + 15) / 16;
  const size_t bytes = (size_t)(256 * (nt * (nt + 1) / 2) + 3 * 16 * nt) * sizeof(double);
  if (NTM > 4) {  // beyond the 64 KB every work-group may have: ask once per device
    static std::atomic<bool> asked[64];
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= 64 || !asked[dev]) {
      hip_check(hipFuncSetAttribute((const void*)k_nw_draw<NTM, W>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)((256 * (NTM * (NTM + 1) / 2) + 3 * 16 * NTM) * sizeof(double))),
                "hipFuncSetAttribute");
      if (dev >= 0 && dev < 64) asked[dev] = true;
    }
  }
  hipLaunchKernelGGL((k_nw_draw<NTM, W>), dim3(1), dim3(64 * W), bytes, s, a);
}

}  // namespace

void launch_nw_draw(const NWArgs& a, hipStream_t s) {
  if (a.K <= 16) launch<1, 4>(a, s);
  else if (a.K <= 32) launch<2, 4>(a, s);
  else if (a.K <= 64) launch<4, 8>(a, s);
  else launch<8, 8>(a, s);
}

}  // namespace mgpu
