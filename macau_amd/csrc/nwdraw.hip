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
// is bound by latency, not by work: a chain of K pivots on one CU.  Tiles cut
// what used to be a barrier (or an LDS round trip) per column or four columns
// to two barriers per 16: the pivots of a diagonal tile run in one wave's
// registers (which also leave U_kk^{-1}, so panels and solves are products),
// the trailing update of the other tiles runs beside the next diagonal tile,
// and the triangular solve needs no barrier at all: a wave owns whole block
// columns of B, and the accumulator layout of a product is the operand layout
// of the next.  Random draws are made beforehand by the work-groups of the
// statistics' reduction, side by side.  Per draw, alone on the card:
//   K                                          10    32    64   100   128
//   one wave's chain (K <= 64), packed
//   triangles in four-column steps (us)        13    41   109   382   588
//   16 x 16 tiles (us)                        5.6   9.9    20    42    48
// At K = 128 (107k cycles): 16k assembling X, 46k factoring, 18k the solve,
// 27k mu and Lambda.
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

// 1/sqrt(d), d > 0: the hardware estimate y (v_rsq_f64, about 23 bits) with one
// third-order step, y (1 + e/2 + 3 e^2 / 8), e = 1 - d y^2 (the next term of
// the series is below 2^-66)
__device__ __forceinline__ double rsqrt_3(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = fma(-d * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
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

// One wave: the diagonal tile X = U U^T, replaced by U^{-1}: the row operations
// that take X to U^T, from the last rows up, take the identity to U^{-1}.
// Four rows at a time, both matrices in the accumulator layout, where register
// v holds rows 4v .. 4v + 3 and is at once the operand of the products that
// these rows enter.  Their 4 x 4 block is broadcast and factored by every lane
// (no lane-to-scalar round trip between its pivots), the rows are multiplied by
// the block's inverse factor E, and the rows above get their rank-4 update:
// 4.9k cycles a tile (bound by the issue of its FP64 instructions), against
// 6.3k with a column of the tile per lane.
// Returns true if a pivot was not positive (it is replaced by 1).
__device__ __forceinline__ bool diag_factor(double* X, int lane) {
  const int lr = lane >> 4, lc = lane & 15;
  f64x4 x = rows(X, lane), id;
#pragma unroll
  for (int v = 0; v < 4; v++) id[v] = 4 * v + lr == lc ? 1.0 : 0.0;
  int bad = 0;
#pragma unroll
  for (int v = 3; v >= 0; v--) {
    double m[4][4], rs[4], E[4][4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int w = 0; w <= u; w++) {
        m[u][w] = rdlane(x[v], 16 * u + 4 * v + w);
        asm volatile("" : "+v"(m[u][w]));  // compares and selects stay on the vector unit
      }
#pragma unroll
    for (int p = 3; p >= 0; p--) {
      const bool ok = m[p][p] > 0.0;
      bad = ok ? bad : 1;
      rs[p] = rsqrt_3(ok ? m[p][p] : 1.0);
#pragma unroll
      for (int i = 0; i < p; i++) m[p][i] *= rs[p];  // u_ip
#pragma unroll
      for (int i = 0; i < p; i++)
#pragma unroll
        for (int w = 0; w <= i; w++) m[i][w] = fma(-m[p][i], m[p][w], m[i][w]);
      // row p of E = (u_ip)^{-1}
      E[p][p] = rs[p];
#pragma unroll
      for (int q = p + 1; q < 4; q++) {
        double t = 0.0;
#pragma unroll
        for (int k = p + 1; k <= q; k++) t = fma(-m[k][p], E[k][q], t);
        E[p][q] = t * rs[p];
      }
    }
    double e = 0.0;  // E[lc][lr]
#pragma unroll
    for (int p = 3; p >= 0; p--)
#pragma unroll
      for (int q = p; q < 4; q++) e = (lc == p && lr == q) ? E[p][q] : e;
    const f64x4 zero = {0.0, 0.0, 0.0, 0.0};
    const double xn = __builtin_amdgcn_mfma_f64_16x16x4f64(e, x[v], zero, 0, 0, 0)[0];
    id[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(e, id[v], zero, 0, 0, 0)[0];
    if (v > 0) {  // rows above: row i takes -u_ip of row p
      const double u = lc < 4 * v ? -xn : 0.0;
      x = __builtin_amdgcn_mfma_f64_16x16x4f64(u, xn, x, 0, 0, 0);
      id = __builtin_amdgcn_mfma_f64_16x16x4f64(u, id[v], id, 0, 0, 0);
    }
  }
  put(X, lane, id);
  return bad != 0;
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
  double* v_m0 = v_w + 16 * nt;   // mu0
  const double kappa_c = a.kappa + a.N;
  const double* S = a.partial + K;
  bool bad = false;

  // 1. X (mvnormal.cpp:322-325; Macau adds lambda_beta beta beta^T to T,
  //    latentprior.cpp:258-260), lower tiles, the entries of T's and S's upper
  //    triangles; the identity beyond K
  constexpr int PER = (NTM * (NTM + 1) / 2 + W - 1) / W;
  f64x4 x[PER];
  int pos[PER];  // the wave's tiles: rows | columns << 16
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int id = min(wave + q * W, ntile - 1);
    int ti = 0;
#pragma unroll
    for (int u = 1; u < NTM; u++) ti += u * (u + 1) / 2 <= id ? 1 : 0;
    pos[q] = ti | (id - ti * (ti + 1) / 2) << 16;
  }
  auto entry = [&](int q, int v, int& r, int& c) {
    r = 16 * (pos[q] & 0xffff) + 4 * v + lr;
    c = 16 * (pos[q] >> 16) + lc;
    return min(min(r, c), K - 1) + min(max(r, c), K - 1) * K;
  };
  f64x4 w[PER];
#pragma unroll
  for (int q = 0; q < PER; q++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      int r, c;
      const int e = entry(q, v, r, c);
      x[q][v] = S[e];
      w[q][v] = a.WI[e];
    }
  for (int k = t; k < 16 * nt; k += 64 * W) {
    const bool in = k < K;
    v_mu[k] = in ? (a.kappa * a.mu0[k] + a.partial[k]) / kappa_c : 0.0;
    v_m0[k] = in ? a.mu0[k] : 0.0;
    v_z[k] = in ? a.bart[KK + k] / sqrt(kappa_c) : 0.0;
  }
  __syncthreads();
  if (a.BBt_partial) {
    const double lb = *a.lambda_beta;
#pragma unroll
    for (int q = 0; q < PER; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        int r, c;
        const int e = entry(q, v, r, c);
        w[q][v] = fma(lb, a.BBt_partial[K + e], w[q][v]);
      }
  }
#pragma unroll
  for (int q = 0; q < PER; q++)
    if (wave + q * W < ntile) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        int r, c;
        entry(q, v, r, c);
        const double y = w[q][v] + x[q][v] + a.kappa * v_m0[r] * v_m0[c] - kappa_c * v_mu[r] * v_mu[c];
        x[q][v] = (r < K && c < K) ? y : (r == c ? 1.0 : 0.0);
      }
      put(X + 256 * (wave + q * W), lane, x[q]);
    }

  // 2. the wave's block column of C^T, on its way while X is factored.  Wave
  //    w takes column w and wave 4 + w column nt - 1 - w, so that the long
  //    and the short columns share a SIMD
  int j = wave < 4 ? wave : nt - 1 - (wave - 4);
  if (wave < 4 ? j >= nt : j < 4) j = nt;  // no column
  f64x4 T[NTM];
#pragma unroll
  for (int q = 0; q < NTM; q++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = 16 * (j + q) + 4 * v + lr, c = 16 * j + lc;
      T[q][v] = a.bart[min(r, K - 1) * K + min(c, K - 1)];
    }
  __syncthreads();

  // 3. X = U U^T, block columns from the last; tile (k, i) below the diagonal
  //    becomes U_ik^T
  for (int k = nt - 1;; k--) {
    if (wave == 0) bad = diag_factor(X + ltile(k, k), lane) || bad;
    __syncthreads();
    if (k == 0) break;
    for (int i = wave; i < k; i += W) {  // U_ik^T = U_kk^{-1} X_ki
      double* P = X + ltile(k, i);
      put(P, lane, mul_add(cols(X + ltile(k, k), lane), rows(P, lane), f64x4{0.0, 0.0, 0.0, 0.0}));
    }
    __syncthreads();
    // X_im -= U_ik U_mk^T: wave 0 takes the next diagonal tile (and goes on
    // to factor it), the others share the rest
    for (int id = wave == 0 ? k * (k + 1) / 2 - 1 : wave - 1; id < k * (k + 1) / 2; id += W - 1) {
      if (wave != 0 && id == k * (k + 1) / 2 - 1) break;
      int i = 0;
      while ((i + 1) * (i + 2) / 2 <= id) i++;
      const int m = id - i * (i + 1) / 2;
      double* P = X + ltile(i, m);
      put(P, lane, mul_add(-rows(X + ltile(k, i), lane), rows(X + ltile(k, m), lane), rows(P, lane)));
      if (wave == 0) break;
    }
    lds_wait();
  }

  // 4. U^T B = C^T, forward, one block column per wave, each step's operands
  //    read from LDS before its products
#pragma unroll
  for (int q = 0; q < NTM; q++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = 16 * (j + q) + 4 * v + lr, c = 16 * j + lc;
      T[q][v] = (r < K && c <= r) ? T[q][v] : (r >= K && r == c ? 1.0 : 0.0);
    }
#pragma unroll
  for (int q = 0; q < NTM; q++)
    if (j + q < nt) {
      const f64x4 d = rows(X + ltile(j + q, j + q), lane);
      f64x4 u[NTM];
#pragma unroll
      for (int p = q + 1; p < NTM; p++) u[p] = cols(X + ltile(min(j + p, nt - 1), j + q), lane);
      T[q] = mul_add(d, T[q], f64x4{0.0, 0.0, 0.0, 0.0});
      const f64x4 minus = -T[q];
#pragma unroll
      for (int p = q + 1; p < NTM; p++)
        if (j + p < nt) T[p] = mul_add(u[p], minus, T[p]);
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
#pragma unroll
    for (int h = 0; h < 2; h++) y[h] *= inv[h];  // x_i once every later row is subtracted
    // 16 rows: their entries of B (over the diagonal) first, then the chain
    auto rows16 = [&](int ti, int top) {
      double b[16][2];
#pragma unroll
      for (int r = 0; r < 16; r++)
#pragma unroll
        for (int h = 0; h <= top; h++) {
          const int i = lane + 64 * h;
          const double v = X[ltile(ti, min(i >> 4, ti)) + tix(r, i & 15)] * inv[h];
          b[r][h] = i < 16 * ti + r ? v : 0.0;
        }
#pragma unroll
      for (int r = 15; r >= 0; r--) {
        const double xr = rdlane(y[top], (16 * ti + r) & 63);
#pragma unroll
        for (int h = 0; h <= top; h++) y[h] = fma(-b[r][h], xr, y[h]);
      }
    };
    if (NTM > 4)
      for (int ti = nt - 1; ti >= 4; ti--) rows16(ti, 1);
    for (int ti = min(nt, 4) - 1; ti >= 0; ti--) rows16(ti, 0);
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int i = lane + 64 * h;
      if (i < K) a.mu[i] = v_mu[i] + y[h];
    }
  } else if (wave == 1) {
    // 6. Lambda mu = B (B^T mu_c + z / sqrt(kappa_c))
    for (int c = lane; c < 16 * nt; c += 64) {
      double s[4] = {v_z[c], 0.0, 0.0, 0.0};
      for (int ti = c >> 4; ti < nt; ti++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[r & 3] += X[ltile(ti, c >> 4) + tix(r, c & 15)] * v_mu[16 * ti + r];
      v_w[c] = (s[0] + s[1]) + (s[2] + s[3]);
    }
    lds_wait();
    for (int r = lane; r < a.KP; r += 64) {
      double s[4] = {0.0, 0.0, 0.0, 0.0};
      if (r < K)
        for (int tj = 0; tj <= r >> 4; tj++)
#pragma unroll
          for (int c = 0; c < 16; c++) s[c & 3] += X[ltile(r >> 4, tj) + tix(r & 15, c)] * v_w[16 * tj + c];
      a.Lmu_f[r] = (float)((s[0] + s[1]) + (s[2] + s[3]));
    }
  } else {
    // 7. Lambda = B B^T, longest tiles first
    int id = 0;
    for (int tj = nt - 1; tj >= 0; tj--)
      for (int ti = tj; ti < nt; ti++, id++) {
        if (id % (W - 2) != wave - 2) continue;
        f64x4 d = {0.0, 0.0, 0.0, 0.0};
        f64x4 u = cols(X + ltile(ti, 0), lane), w = cols(X + ltile(tj, 0), lane);
        for (int k = 0; k <= tj; k++) {  // the next operands on their way under the products
          const int kn = min(k + 1, tj);
          const f64x4 un = cols(X + ltile(ti, kn), lane), wn = cols(X + ltile(tj, kn), lane);
          d = mul_add(u, w, d);
          u = un;
          w = wn;
        }
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
  const size_t bytes = (size_t)(256 * (nt * (nt + 1) / 2) + 4 * 16 * nt) * sizeof(double);
  if (NTM > 4) {  // beyond the 64 KB every work-group may have: ask once per device
    static std::atomic<bool> asked[64];
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= 64 || !asked[dev]) {
      hip_check(hipFuncSetAttribute((const void*)k_nw_draw<NTM, W>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)((256 * (NTM * (NTM + 1) / 2) + 4 * 16 * NTM) * sizeof(double))),
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
