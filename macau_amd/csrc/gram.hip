// gram.hip -- the link-matrix updates on F's non-empty columns.
//
// Side information with many features often has most of its columns empty
// (hashed or enumerated fingerprints).
//
// * Block CG (linop.h:228-343).  K = F^T F + reg I is reg I on the empty columns,
//   where every iterate is therefore a combination C R0 of the rows of its
//   starting residual R0, with the nr x nr coefficients C common to all of them.
//   Inner products over them see R0 only through R0 R0^T = W W^T, so they are
//   replaced by the nr columns of the Cholesky factor W: the iteration runs on
//   n + nr features (n non-empty ones) with the same inner products, hence the
//   same coefficients, residual norms and iteration count (up to rounding), and
//   the empty features get X = X_v W^{-1} R0 at the end.
// * The Gram matrix G = F^T F of the non-empty columns (n x n FP64) is formed once,
//   when the prior is set up, where that pays (gram_for_sweep, gram_for_cg); block
//   CG's products F^T (F P) then become G P.
// * The univariate sweep (macauoneprior.cpp:215-252) on G.  A feature's update
//   needs F_f . z, and changes z by a multiple of F_f: on c = F^T z the change is
//   a column of G.  A latent's chain is then one broadcast and one multiply-add
//   per feature, 64 features at a time on one wave, with the rest of c updated by
//   products; it no longer walks the columns' entries.
//
// Measured at 15000 rows: the sweep of 32 latents over 969 non-empty columns with
// about 900 entries each 2.9 -> 0.6 ms an iteration (bound by the chain, 0.25 us a
// feature, and G's reads); block CG with 100000 columns, 5700 of them non-empty,
// 137 -> 95 us a CG iteration (bound by F's products and the small solves).
#include <algorithm>

#include "common.h"
#include "model.h"

namespace mgpu {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// --- G ---

// rows [r0, r0 + nr) of F over the non-empty columns, dense (np doubles a row,
// zero on entry); a thread per row, entries in order
__global__ void __launch_bounds__(256) k_gram_rows(CsrDev F, const int* __restrict__ pos, int np, int r0, int nr,
                                                   double* __restrict__ D) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= nr) return;
  double* d = D + (size_t)r * np;
  for (int e = F.row_ptr[r0 + r]; e < F.row_ptr[r0 + r + 1]; e++) {
    const int j = F.cols[e];
    d[pos ? pos[j] : j] += F.vals ? F.vals[e] : 1.0;
  }
}

// part[s][tile] (+)= D^T D over the s-th share of the rows: a work-group per 64
// x 64 tile (i >= j) and share, a 32 x 32 quadrant per wave, four rows per
// matrix instruction, operands straight from global memory
__global__ void __launch_bounds__(256) k_gram_tiles(const double* __restrict__ D, int np, int nr, int ntile,
                                                    int first, double* __restrict__ part) {
  int ti = 0;
  while ((ti + 1) * (ti + 2) / 2 <= (int)blockIdx.x) ti++;
  const int tj = blockIdx.x - ti * (ti + 1) / 2;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int i0 = 64 * ti + 32 * (w >> 1) + c, j0 = 64 * tj + 32 * (w & 1) + c;
  const int per = (nr / 16 + gridDim.y - 1) / gridDim.y * 16;  // nr is a multiple of 16
  const int b = min(nr, (int)blockIdx.y * per), e = min(nr, b + per);
  double* out = part + ((size_t)blockIdx.y * ntile + blockIdx.x) * 4096 + w * 1024;
  f64x4 acc[2][2];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int q = 0; q < 4; q++) acc[u][v][q] = first ? 0.0 : out[(2 * u + v) * 256 + 64 * q + lane];
  for (int r = b; r < e; r += 16) {
    double x[4][2], y[4][2];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const double* d = D + (size_t)(r + 4 * s + g) * np;
      x[s][0] = d[i0];
      x[s][1] = d[i0 + 16];
      y[s][0] = d[j0];
      y[s][1] = d[j0 + 16];
    }
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++)
          acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s][u], y[s][v], acc[u][v], 0, 0, 0);
  }
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int q = 0; q < 4; q++) out[(2 * u + v) * 256 + 64 * q + lane] = acc[u][v][q];
}

// G = the shares' tiles summed in order, both triangles
__global__ void __launch_bounds__(256) k_gram_sum(const double* __restrict__ part, int np, int ntile, int nshare,
                                                  double* __restrict__ G) {
  int ti = 0;
  while ((ti + 1) * (ti + 2) / 2 <= (int)blockIdx.x) ti++;
  const int tj = blockIdx.x - ti * (ti + 1) / 2;
  for (int q = threadIdx.x; q < 4096; q += 256) {
    double s = 0.0;
    for (int b = 0; b < nshare; b++) s += part[((size_t)b * ntile + blockIdx.x) * 4096 + q];
    const int w = q >> 10, t = q >> 8 & 3, r = q >> 4 & 15, c = q & 15;
    const int i = 64 * ti + 32 * (w >> 1) + 16 * (t >> 1) + r, j = 64 * tj + 32 * (w & 1) + 16 * (t & 1) + c;
    G[(size_t)i * np + j] = s;
    G[(size_t)j * np + i] = s;
  }
}

// --- block CG ---

// KP = G P + reg P on the n + nv compact features (reg P on the nv last):
// 16 features per work-group, G's columns shared by the four waves, their sums
// added in order through LDS.  Bound by the launch and the matrix chain (n / 16
// dependent steps per wave).
template <int NT>  // 16-component tiles of the right-hand sides
__global__ void __launch_bounds__(256) k_gram_mm(const double* __restrict__ G, int np, int n, int ntot, int nr,
                                                 const double* __restrict__ P, const double* __restrict__ reg,
                                                 double* __restrict__ KP, const double* __restrict__ skip) {
  if (*skip != 0.0) return;
  __shared__ double red[4][NT][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int i0 = 16 * blockIdx.x;
  f64x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f64x4{0.0, 0.0, 0.0, 0.0};
  if (i0 < n) {
    const int per = ((n + 3) / 4 + 15) / 16 * 16, b = min(n, w * per), e = min(n, b + per);
    for (int k = b; k < e; k += 16) {
      double x[4], y[4][NT];
#pragma unroll
      for (int s = 0; s < 4; s++) {
        // (rows of G from n on are zero, up to np; P has rows past n)
        const int r = k + 4 * s + g;
        x[s] = G[(size_t)min(r, np - 1) * np + i0 + c];
#pragma unroll
        for (int t = 0; t < NT; t++) y[s][t] = 16 * t + c < nr ? P[(size_t)min(r, ntot - 1) * nr + 16 * t + c] : 0.0;
      }
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int t = 0; t < NT; t++)
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(k + 4 * s + g < n ? x[s] : 0.0, y[s][t], acc[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int v = 0; v < 4; v++) red[w][t][64 * v + lane] = acc[t][v];
  __syncthreads();
  const double lam = *reg;
  const int f = i0 + (threadIdx.x >> 4);
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int i = 16 * t + (threadIdx.x & 15);
    if (f < ntot && i < nr) {
      const double s = ((red[0][t][threadIdx.x] + red[1][t][threadIdx.x]) + red[2][t][threadIdx.x]) +
                       red[3][t][threadIdx.x];
      KP[(size_t)f * nr + i] = s + lam * P[(size_t)f * nr + i];
    }
  }
}

// The compact right-hand side: B's non-empty columns, then (work-group 0) the
// columns of W, S = W W^T the sum over the empty features.  A pivot below 1e-12
// of its diagonal entry raises *bad: W is taken as zero (the iteration then runs
// on the non-empty columns alone), and the others are solved as B / reg.
__global__ void __launch_bounds__(256) k_gram_begin(const double* __restrict__ S, const double* __restrict__ B,
                                                    const int* __restrict__ idx, int n, int nr,
                                                    double* __restrict__ Bc, double* __restrict__ W, double* bad) {
  const int t = threadIdx.x;
  if (blockIdx.x > 0) {
    for (size_t q = (size_t)(blockIdx.x - 1) * 256 + t; q < (size_t)n * nr; q += (size_t)(gridDim.x - 1) * 256)
      Bc[q] = B[(size_t)idx[q / nr] * nr + q % nr];
    return;
  }
  __shared__ double A[32][33];
  __shared__ double d0[32];
  const int i = t & 31, j0 = t >> 5;
  for (int j = j0; j < nr; j += 8)
    if (i < nr) A[i][j] = S[i + j * nr];
  if (t < nr) d0[t] = S[t + t * nr];
  __syncthreads();
  bool fail = false;
  for (int k = 0; k < nr; k++) {
    const double d = A[k][k];
    const bool ok = d > 1e-12 * d0[k];
    fail = fail || !ok;
    const double rs = 1.0 / sqrt(ok ? d : 1.0);
    const double aik = i < nr && i >= k ? A[i][k] * rs : 0.0;
    __syncthreads();
    if (j0 == 0 && i < nr && i >= k) A[i][k] = aik;
    __syncthreads();
    for (int j = k + 1 + j0; j < nr; j += 8)
      if (i < nr && i >= j) A[i][j] -= aik * A[j][k];
    __syncthreads();
  }
  for (int j = j0; j < nr; j += 8)
    if (i < nr) {
      const double w = i >= j && !fail ? A[i][j] : 0.0;
      W[i + j * nr] = w;
      Bc[(size_t)(n + j) * nr + i] = w;
    }
  if (t == 0) *bad = fail ? 1.0 : 0.0;
}

// M = X_v W^{-1} (nr x nr, col-major; the identity over reg when *bad); a row
// per lane, from the last column
__global__ void __launch_bounds__(64) k_gram_coef(const double* __restrict__ Xc, const double* __restrict__ W,
                                                  const double* bad, const double* reg, int n, int nr,
                                                  double* __restrict__ M) {
  if (*bad != 0.0) {
    for (int q = threadIdx.x; q < nr * nr; q += 64) M[q] = q % nr == q / nr ? 1.0 / *reg : 0.0;
    return;
  }
  __shared__ double w[32][33];
  const int i = threadIdx.x;
  for (int q = i; q < 32 * 32; q += 64) {
    const int r = q & 31, c = q >> 5;
    w[r][c] = r < nr && c < nr ? W[r + c * nr] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  if (i >= nr) return;
  double x[32];
#pragma unroll
  for (int j = 0; j < 32; j++) x[j] = j < nr ? Xc[(size_t)(n + j) * nr + i] : 0.0;
#pragma unroll
  for (int j = 31; j >= 0; j--) {
    x[j] /= w[j][j];
#pragma unroll
    for (int k = 0; k < j; k++) x[k] -= x[j] * w[j][k];
  }
#pragma unroll
  for (int j = 0; j < 32; j++)
    if (j < nr) M[i + j * nr] = x[j];
}

// X = Xc on the non-empty features, M B on the others: 16 features per wave and
// step, M in registers as the left operand (component 4 (m % 4) + m / 4 of a
// 16-block on its row m, so that a lane's results are four neighbours), the
// reduction index dealt so that a lane's share of B is contiguous
__global__ void __launch_bounds__(256) k_gram_expand(const double* __restrict__ M, const double* __restrict__ Xc,
                                                     const int* __restrict__ pos, const double* __restrict__ B,
                                                     int nfeat, int nr, double* __restrict__ X) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  double m[2][8];
#pragma unroll
  for (int rb = 0; rb < 2; rb++)
#pragma unroll
    for (int s = 0; s < 8; s++) {
      const int i = 16 * rb + 4 * (c & 3) + (c >> 2), k = 8 * g + s;
      m[rb][s] = i < nr && k < nr ? M[i + k * nr] : 0.0;
    }
  const int nt = (nfeat + 15) / 16;
  for (int t = blockIdx.x * 4 + (threadIdx.x >> 6); t < nt; t += gridDim.x * 4) {
    const int f = 16 * t + c, fc = min(f, nfeat - 1);
    const int p = pos[fc];
    const double* b = B + (size_t)fc * nr;
    double y[8];
#pragma unroll
    for (int s = 0; s < 8; s++) y[s] = 8 * g + s < nr ? b[8 * g + s] : 0.0;
    f64x4 d[2];
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
      d[rb] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 8; s++) d[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(m[rb][s], y[s], d[rb], 0, 0, 0);
    }
    if (f < nfeat) {
#pragma unroll
      for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int i = 16 * rb + 4 * g + v;
          if (i < nr) X[(size_t)f * nr + i] = p >= 0 ? Xc[(size_t)p * nr + i] : d[rb][v];
        }
    }
  }
}

// --- univariate sweep ---

// Z = U - mu - Uhat (K x N, FP64)
__global__ void __launch_bounds__(256) k_uni_resid(BetaUniArgs a, double* __restrict__ Z) {
  const size_t tot = (size_t)a.N * a.K;
  for (size_t q = (size_t)blockIdx.x * 256 + threadIdx.x; q < tot; q += (size_t)gridDim.x * 256) {
    const int n = (int)(q / a.K), d = (int)(q % a.K);
    Z[q] = (double)a.U[(size_t)n * a.KP + d] - a.mu[d] - a.uhat[q];
  }
}

// One latent per work-group.  c = F^T z over the non-empty features; feature f
// in order gives beta_f = (lambda (c_f + beta_f |F_f|^2)) / A_f + its normal and
// c += G[:, f] (beta_f old - new).  64 features at a time: on wave 0, lane i
// holding feature i of the block (its step is linear in c_f, so every lane
// keeps its own next value and a step is a broadcast and a multiply-add; 16
// steps' columns of G are loaded ahead), then the rest of c as products, a
// 64-entry share per wave at a time.
constexpr int kSweepWaves = 8;
__global__ void __launch_bounds__(64 * kSweepWaves) k_uni_sweep(BetaUniArgs a, GramPlan gp,
                                                                const double* __restrict__ Fz) {
  __shared__ double c[kGramMax], del[64];
  const int d = blockIdx.x, t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int K = a.K, n = gp.n, np = gp.np, nb = (n + 63) / 64;
  const double lam = a.Lambda[d + d * K];
  for (int q = t; q < 64 * nb; q += 64 * kSweepWaves) c[q] = q < n ? Fz[(size_t)gp.idx[q] * K + d] : 0.0;
  __syncthreads();
  for (int r = 0; r < nb; r++) {
    const double* Gr = gp.G + (size_t)64 * r * np;
    if (w == 0) {
      const int i = 64 * r + lane;
      const bool in = i < n;
      const int f = gp.idx[in ? i : n - 1];
      const double bo = a.beta[(size_t)f * K + d], ai = a.ainv[(size_t)d * a.nfeat + f];
      const double a1 = in ? lam * ai : 0.0;
      const double d0 = in ? bo - fma(lam * (bo * a.colsq[f]), ai, a.nz[(size_t)d * a.nfeat + f]) : 0.0;
      double cv = c[i], mine = 0.0, x[2][16];
      auto load = [&](double(&v)[16], int s0) {
#pragma unroll
        for (int s = 0; s < 16; s++) v[s] = Gr[(size_t)(s0 + s) * np + 64 * r + lane];
      };
      auto steps = [&](const double(&v)[16], int s0) {
#pragma unroll
        for (int s = 0; s < 16; s++) {
          const double dv = fma(-cv, a1, d0);  // old - new of this lane's feature, were it its turn
          mine = lane == s0 + s ? dv : mine;
          cv = fma(v[s], rdlane(dv, s0 + s), cv);
        }
      };
      load(x[0], 0);
      load(x[1], 16);
      steps(x[0], 0);
      load(x[0], 32);
      steps(x[1], 16);
      load(x[1], 48);
      steps(x[0], 32);
      steps(x[1], 48);
      del[lane] = mine;
      if (in) a.beta[(size_t)f * K + d] = bo - mine;
    }
    __syncthreads();
    for (int q = r + 1 + w; q < nb; q += kSweepWaves) {
      double s[4] = {c[64 * q + lane], 0.0, 0.0, 0.0};
#pragma unroll 16
      for (int u = 0; u < 64; u++) s[u & 3] = fma(Gr[(size_t)u * np + 64 * q + lane], del[u], s[u & 3]);
      c[64 * q + lane] = (s[0] + s[1]) + (s[2] + s[3]);
    }
    __syncthreads();
  }
}

}  // namespace

void launch_gram(const CsrDev& F, bool compact, const GramPlan& g, double* G, hipStream_t s) {
  const int nb = g.np / 64, ntile = nb * (nb + 1) / 2;
  const int shares = std::max(1, std::min(16, 512 / ntile));
  // dense rows at most 128 MB at a time
  const int chunk = std::max(64, std::min((F.nrow + 15) / 16 * 16, (int)((128 << 20) / ((size_t)g.np * 8)) / 16 * 16));
  DevBuf D((size_t)chunk * g.np * sizeof(double)), part((size_t)shares * ntile * 4096 * sizeof(double));
  for (int r0 = 0; r0 < F.nrow; r0 += chunk) {
    const int nr = std::min(chunk, F.nrow - r0), nrp = (nr + 15) / 16 * 16;
    HIPCHK(hipMemsetAsync(D.as<void>(), 0, (size_t)nrp * g.np * sizeof(double), s));
    hipLaunchKernelGGL(k_gram_rows, dim3((nr + 255) / 256), dim3(256), 0, s, F, compact ? nullptr : g.pos, g.np, r0, nr,
                       D.as<double>());
    hipLaunchKernelGGL(k_gram_tiles, dim3(ntile, shares), dim3(256), 0, s, (const double*)D.as<double>(), g.np, nrp,
                       ntile, r0 == 0 ? 1 : 0, part.as<double>());
  }
  hipLaunchKernelGGL(k_gram_sum, dim3(ntile), dim3(256), 0, s, (const double*)part.as<double>(), g.np, ntile, shares,
                     G);
  HIPCHK(hipStreamSynchronize(s));  // the transient buffers go out of scope
}

void launch_gram_mm(const GramPlan& g, int ntot, int nr, const double* P, const double* reg, double* KP,
                    const double* skip, hipStream_t s) {
  const dim3 grid((ntot + 15) / 16);
  if (nr <= 16) hipLaunchKernelGGL(k_gram_mm<1>, grid, dim3(256), 0, s, g.G, g.np, g.n, ntot, nr, P, reg, KP, skip);
  else hipLaunchKernelGGL(k_gram_mm<2>, grid, dim3(256), 0, s, g.G, g.np, g.n, ntot, nr, P, reg, KP, skip);
}

void launch_gram_begin(const GramPlan& g, const double* S, const double* B, int nr, double* Bc, double* W, double* bad,
                       hipStream_t s) {
  const int blocks = 1 + std::max(1, std::min(256, (g.n * nr + 1023) / 1024));
  hipLaunchKernelGGL(k_gram_begin, dim3(blocks), dim3(256), 0, s, S, B, g.idx, g.n, nr, Bc, W, bad);
}

void launch_gram_end(const GramPlan& g, const double* Xc, const double* W, const double* bad, const double* reg,
                     const double* B, int nfeat, int nr, double* M, double* X, hipStream_t s) {
  hipLaunchKernelGGL(k_gram_coef, dim3(1), dim3(64), 0, s, Xc, W, bad, reg, g.n, nr, M);
  const int blocks = std::max(1, std::min(2048, (nfeat + 63) / 64));
  hipLaunchKernelGGL(k_gram_expand, dim3(blocks), dim3(256), 0, s, (const double*)M, Xc, g.pos, B, nfeat, nr, X);
}

void launch_uni_resid(const BetaUniArgs& a, double* Z, hipStream_t s) {
  const size_t tot = (size_t)a.N * a.K;
  const unsigned grid = (unsigned)std::max<size_t>(1, std::min<size_t>(4096, (tot + 255) / 256));
  hipLaunchKernelGGL(k_uni_resid, dim3(grid), dim3(256), 0, s, a, Z);
}

void launch_uni_sweep(const BetaUniArgs& a, const GramPlan& g, const double* Fz, hipStream_t s) {
  hipLaunchKernelGGL(k_uni_sweep, dim3(a.K), dim3(64 * kSweepWaves), 0, s, a, g, Fz);
}

}  // namespace mgpu
