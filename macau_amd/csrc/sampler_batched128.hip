// sampler_batched128.hip -- the batched per-row sampler for K in (64, 128]:
// split-BF16 MFMA Gram of a 128 x 128 precision matrix, one row per wave (up to
// 1024 rows: two, four or eight waves share its Gram, k_light128w).
//
// Same mathematics as the K <= 64 samplers (sample_latent_blas,
// latentprior.cpp:361-385): P = Lambda + alpha G = L L^T, b = alpha c +
// Lambda mu, u = L^{-T}(L^{-1} b + z); rows above the segment length are split
// into segments whose partial Grams are summed in segment order; light rows are
// taken by decreasing nnz.
//
// A wave holds the row's whole matrix: 36 tiles (16 x 16) of the upper
// triangle (P = R^T R, R = L^T) in the accumulator layout of
// v_mfma_f32_16x16x*: lane (g, n) = (l / 16, l % 16) has in register v the
// entry of hardware row 4g + v, column n.  Component sigma(h) = 4 (h % 4) + h / 4
// of a 16-block sits at hardware index h, so register v holds components 4v + g
// of the rows: a register is then at once the operand (four consecutive rows)
// of the product that these rows enter, and the factorisation and both solves
// run on registers alone.  LDS holds only Lambda (one copy for the work-group's
// eight waves, in tiles), a 1 KB transposition buffer per wave, and the normals.
//   * Gram: per 32-nonzero chunk lane (g, n) gathers component sigma(n) of each
//     block of nonzeros 8g .. 8g + 7, which is the operand layout of
//     v_mfma_f32_16x16x32_bf16.  A factor enters in three BF16 parts (24 bits),
//     a tile takes six of their nine products: HiHi^T + HiMid^T + MidHi^T +
//     MidMid^T + HiLo^T + LoHi^T.
//   * Factorisation by 16 columns: the diagonal tile gives L_kk^{-1} (see
//     diag_factor), row k's tiles become R_kj = L_kk^{-1} P_kj and the rest
//     P_ij -= R_ki^T R_kj.
//   * Solves by 16 components: products of tiles and vectors, the sums over
//     lanes taken once per block.
//   * Component blocks beyond K are neither gathered, nor updated, nor solved.
//   * No condition probes: refinement is not offered at this size.
// Segments (k_seg128) share a segment's Gram between four waves through LDS.
#include <algorithm>
#include <stdexcept>

#include "batched.h"

namespace mgpu {

namespace {

constexpr int kThreads128 = 256;
constexpr int kTiles = 36;                        // 16 x 16 tiles of the upper triangle
constexpr int kPartial128 = kTiles * 256 + 128;   // floats per segment partial: tiles and RHS sums

__device__ __forceinline__ int sigma(int h) { return 4 * (h & 3) + (h >> 2); }
__device__ __forceinline__ constexpr int slot(int i, int j) { return j * (j + 1) / 2 + i; }  // tile (i, j), i <= j

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int NO>
struct Lds128 {               // of the segment kernel
  uint4 op[2][8][64][3];      // Gram operands: [buffer][component block][lane][hi, mid, lo]
  i32x4 ix[4][NO][8];         // each wave's copy of the chunk's indices
  f32x4 r[4][8];              // and residuals
};

__device__ __forceinline__ f32x4 mul_add(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int s = 0; s < 4; s++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], c, 0, 0, 0);
  return c;
}

// sum over the 16 lanes of a row of lanes
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __builtin_bit_cast(
                 float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum16(float x) {
  x = dpp_add<0x128>(x);  // row_ror:8, 4, 2, 1
  x = dpp_add<0x124>(x);
  x = dpp_add<0x122>(x);
  return dpp_add<0x121>(x);
}
// sum over the four rows of lanes
__device__ __forceinline__ float sum_rows(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// The diagonal tile x = L L^T: the row operations that take it to L^T, from
// the first rows down, take the identity to L^{-1}, which is returned.  Four
// rows (one register) at a time: their 4 x 4 block is broadcast and factored by
// every lane, the rows are multiplied by the block's inverse factor E, and the
// rows below get their rank-4 update.  A pivot that is not positive raises bad
// and is replaced by 1.
__device__ __forceinline__ f32x4 diag_factor(f32x4 x, int lane, int& bad) {
  const int g = lane >> 4, n = lane & 15;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 id;
#pragma unroll
  for (int v = 0; v < 4; v++) id[v] = 4 * v + g == sigma(n) ? 1.f : 0.f;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    float m[4][4], rs[4], E[4][4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int w = 0; w <= u; w++) {
        m[u][w] = rdlane(x[v], 16 * u + 4 * w + v);
        asm volatile("" : "+v"(m[u][w]));  // compares and selects stay on the vector unit
      }
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const bool ok = m[p][p] > 0.f;
      bad = ok ? bad : 1;
      rs[p] = __builtin_amdgcn_rsqf(ok ? m[p][p] : 1.f);
#pragma unroll
      for (int i = p + 1; i < 4; i++) m[i][p] *= rs[p];
#pragma unroll
      for (int i = p + 1; i < 4; i++)
#pragma unroll
        for (int w = p + 1; w <= i; w++) m[i][w] = fmaf(-m[i][p], m[w][p], m[i][w]);
      E[p][p] = rs[p];
#pragma unroll
      for (int q = 0; q < p; q++) {
        float t = 0.f;
#pragma unroll
        for (int k = q; k < p; k++) t = fmaf(-m[p][k], E[k][q], t);
        E[p][q] = t * rs[p];
      }
    }
    float e = 0.f;  // left operand: E's row n / 4 at hardware row n = 0, 4, 8, 12
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
      for (int q = 0; q <= p; q++) e = (n == 4 * p && g == q) ? E[p][q] : e;
    const float xn = __builtin_amdgcn_mfma_f32_16x16x4f32(e, x[v], zero, 0, 0, 0)[0];
    id[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(e, id[v], zero, 0, 0, 0)[0];
    if (v < 3) {
      const float u = (n & 3) > v ? -xn : 0.f;  // the rows below
      x = __builtin_amdgcn_mfma_f32_16x16x4f32(u, xn, x, 0, 0, 0);
      id = __builtin_amdgcn_mfma_f32_16x16x4f32(u, id[v], id, 0, 0, 0);
    }
  }
  return id;
}

// Gram stream over the nonzeros of one segment, shared by four waves: wave w
// gathers component blocks 2w and 2w + 1 and splits them into LDS
// (double-buffered, one barrier per chunk, the next chunk's gathers under this
// chunk's products); the tiles are shared out by operand reuse: 10 + 10 of the
// two diagonal quadrants, 8 + 8 of the third.
template <int NO>
struct Gram128 {
  const SampleArgs& a;
  const Factors<NO>& F;
  Lds128<NO>& s;
  const int nt, lane, w, g, cn;
  int beg = 0, end = 0;
  int ixr[NO];
  float rr;
  float v[2][8];  // component 32w + 16h + cn of the lane's nonzeros of the chunk

  __device__ Gram128(const SampleArgs& a_, const Factors<NO>& F_, Lds128<NO>& s_, int nt_)
      : a(a_), F(F_), s(s_), nt(nt_), lane(threadIdx.x & 63), w(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)),
        g(lane >> 4), cn(sigma(lane & 15)) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int q = 0; q < 8; q++) v[h][q] = 0.f;
  }
  // indices and residual of nonzero e0 + lane, lanes 0..31 (index -1: none)
  __device__ __forceinline__ void load_ix(int e0) {
    const int e = e0 + (lane & 31);
    const bool ok = e < end;
#pragma unroll
    for (int t = 0; t < NO; t++) ixr[t] = ok ? a.rows.idx[(size_t)e * NO + t] : -1;
    rr = ok ? a.rows.r[e] : 0.f;
  }
  // their copy in LDS, and the chunk's factor values on their way
  __device__ __forceinline__ void gather() {
    if (lane < 32) {
#pragma unroll
      for (int t = 0; t < NO; t++) reinterpret_cast<int*>(s.ix[w][t])[lane] = ixr[t];
      reinterpret_cast<float*>(s.r[w])[lane] = rr;
    }
    lds_wait();
#pragma unroll
    for (int t = 0; t < NO; t++) {
      const i32x4 ix[2] = {s.ix[w][t][2 * g], s.ix[w][t][2 * g + 1]};
#pragma unroll
      for (int h = 0; h < 2; h++) {
        if (2 * w + h >= nt) continue;
#pragma unroll
        for (int q = 0; q < 8; q++) {
          const float x = ld_factor<128>(F.rs[t], ix[q >> 2][q & 3], 32 * w + 16 * h + cn);
          v[h][q] = t == 0 ? x : v[h][q] * x;
        }
      }
    }
  }
  // the indices of [b, e)'s first chunk, then its values
  __device__ __forceinline__ void open(int b, int e) {
    beg = b;
    end = e;
    load_ix(beg);
  }
  __device__ __forceinline__ void start() {
    gather();
    load_ix(beg + 32);
  }
  // acc: the tiles of the wave's quarter (see gram_tiles), sums: the RHS sums
  // of blocks 2w and 2w + 1, partial over the lane's nonzeros
  __device__ __forceinline__ void run(f32x4 (&acc)[10], float (&sums)[2]) {
#pragma unroll
    for (int q = 0; q < 10; q++) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    sums[0] = sums[1] = 0.f;
    const int nch = (end - beg + 31) >> 5;
    for (int c = 0; c < nch; c++) {
      const int buf = c & 1;
      {
        const f32x4 r[2] = {s.r[w][2 * g], s.r[w][2 * g + 1]};
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
          for (int q = 0; q < 8; q++) sums[h] += v[h][q] * r[q >> 2][q & 3];
          bf16x8 x[3];
          split8(v[h], x[0], x[1], x[2]);
#pragma unroll
          for (int t = 0; t < 3; t++) s.op[buf][2 * w + h][lane][t] = __builtin_bit_cast(uint4, x[t]);
        }
      }
      __syncthreads();
      if (c + 1 < nch) {
        gather();
        load_ix(beg + 32 * (c + 2));
      }
      auto op = [&](int I, bf16x8 (&x)[3]) {
#pragma unroll
        for (int t = 0; t < 3; t++) x[t] = __builtin_bit_cast(bf16x8, s.op[buf][I][lane][t]);
      };
      auto product = [&](f32x4& d, const bf16x8 (&x)[3], const bf16x8 (&y)[3]) {
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
          for (int u = 0; u < 3 - t; u++) d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t], y[u], d, 0, 0, 0);
      };
      // the wave's columns J, and its rows: the quadrant's diagonal (waves 0,
      // 1) or rows 0-1 / 2-3 (waves 2, 3) against columns 4-7
      const int J0 = w == 0 ? 0 : 4;
      bf16x8 y[4][3];
#pragma unroll
      for (int j = 0; j < 4; j++) op(J0 + j, y[j]);
      if (w < 2) {
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (J0 + j < nt) {
#pragma unroll
            for (int i = 0; i <= j; i++) product(acc[j * (j + 1) / 2 + i], y[i], y[j]);
          }
      } else {
#pragma unroll
        for (int i = 0; i < 2; i++) {
          bf16x8 x[3];
          op(2 * (w - 2) + i, x);
#pragma unroll
          for (int j = 0; j < 4; j++)
            if (4 + j < nt) product(acc[4 * i + j], x, y[j]);
        }
      }
    }
  }
};

// f(q, i, j) for the Gram tiles of wave w in the first nt component blocks
template <typename F>
__device__ __forceinline__ void gram_tiles(int w, int nt, F&& f) {
  if (w < 2) {
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (4 * w + j < nt) {
#pragma unroll
        for (int i = 0; i <= j; i++) f(j * (j + 1) / 2 + i, 4 * w + i, 4 * w + j);
      }
  } else {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (4 + j < nt) f(4 * i + j, 2 * (w - 2) + i, 4 + j);
  }
}

// What the waves of a light- or heavy-row work-group share.
constexpr int kWaves128 = 8;
template <int NO, int NT>
struct Shared128 {
  f32x4 lam[slot(0, NT)][64];            // Lambda, in tiles
  struct Wave {
    f32x4 t[64];                     // transposition of L_kk^{-1}
    f32x4 v[8][4];                   // the normals, then u: [block][g], register v = component 4v + g
    i32x4 ix[NO][8];                 // the chunk's indices
    f32x4 r[8];                      // and residuals
    uint4 lo[NT][64];                // and the factors' low parts
  } wave[kWaves128];
};

template <int NO, int NT>
__device__ __forceinline__ void load_lambda(const SampleArgs& a, Shared128<NO, NT>& s) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int q = w; q < slot(0, NT); q += kWaves128) {
    int j = 0;
    while (slot(0, j + 1) <= q) j++;
    const float* l = a.Lambda_f + (16 * (q - slot(0, j)) + (lane >> 4)) * 128 + 16 * j + sigma(lane & 15);
    f32x4 x;
#pragma unroll
    for (int v = 0; v < 4; v++) x[v] = l[4 * v * 128];
    s.lam[q][lane] = x;
  }
  __syncthreads();
}

// One wave: the Gram tiles of the nonzeros [beg, end) and the RHS sums c
// (component 16 I + sigma(n) of block I, on every row of lanes).
template <int NO, int NT>
__device__ __forceinline__ void gram_row(const SampleArgs& a, const Factors<NO>& F, typename Shared128<NO, NT>::Wave& s,
                                         int beg, int end, f32x4 (&P)[slot(0, NT)], float (&c)[NT]) {
  const int lane = threadIdx.x & 63, g = lane >> 4, cn = sigma(lane & 15);
#pragma unroll
  for (int q = 0; q < slot(0, NT); q++) P[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int I = 0; I < NT; I++) c[I] = 0.f;
  int ixr[NO];
  float rr;
  auto load_ix = [&](int e0) {
    const int e = e0 + (lane & 31);
    const bool ok = e < end;
#pragma unroll
    for (int t = 0; t < NO; t++) ixr[t] = ok ? a.rows.idx[(size_t)e * NO + t] : -1;
    rr = ok ? a.rows.r[e] : 0.f;
  };
  load_ix(beg);
  for (int e0 = beg; e0 < end; e0 += 32) {
    if (lane < 32) {
#pragma unroll
      for (int t = 0; t < NO; t++) reinterpret_cast<int*>(s.ix[t])[lane] = ixr[t];
      reinterpret_cast<float*>(s.r)[lane] = rr;
    }
    lds_wait();
    i32x4 ix[NO][2];
#pragma unroll
    for (int t = 0; t < NO; t++) {
      ix[t][0] = s.ix[t][2 * g];
      ix[t][1] = s.ix[t][2 * g + 1];
    }
    const f32x4 r[2] = {s.r[2 * g], s.r[2 * g + 1]};
    load_ix(e0 + 32);
    int at[NO][8];
#pragma unroll
    for (int t = 0; t < NO; t++)
#pragma unroll
      for (int q = 0; q < 8; q++) at[t][q] = factor_at<128>(ix[t][q >> 2][q & 3], cn);
    bf16x8 hi[NT], mid[NT];
#pragma unroll
    for (int I = 0; I < NT; I++) {
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        v[q] = ld_at(F.rs[0], at[0][q], 16 * I);
#pragma unroll
        for (int t = 1; t < NO; t++) v[q] *= ld_at(F.rs[t], at[t][q], 16 * I);
        c[I] = fmaf(v[q], r[q >> 2][q & 3], c[I]);
      }
      bf16x8 lo;
      split8(v, hi[I], mid[I], lo);
      s.lo[I][lane] = __builtin_bit_cast(uint4, lo);
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
#pragma unroll
      for (int i = 0; i < NT; i++) {
        if (i > j) continue;
        f32x4& d = P[slot(i, j)];
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi[i], hi[j], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi[i], mid[j], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mid[i], hi[j], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mid[i], mid[j], d, 0, 0, 0);
      }
    }
#pragma unroll
    for (int k = 0; k < NT; k++) {
      const bf16x8 lo = __builtin_bit_cast(bf16x8, s.lo[k][lane]);
#pragma unroll
      for (int i = 0; i <= k; i++)
        P[slot(i, k)] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi[i], lo, P[slot(i, k)], 0, 0, 0);
#pragma unroll
      for (int j = k; j < NT; j++)
        P[slot(k, j)] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, hi[j], P[slot(k, j)], 0, 0, 0);
    }
  }
#pragma unroll
  for (int I = 0; I < NT; I++) c[I] = sum_rows(c[I]);
}

// One wave: the row's sample from its Gram tiles and RHS sums; returns the
// lane's share of the train SSE (when sse_partial is set).
template <int NO, int NT>
__device__ __forceinline__ double finish_row(const SampleArgs& a, int row, int it, float alpha, const f32x4 (*lam)[64],
                                             typename Shared128<NO, NT>::Wave& s, f32x4 (&P)[slot(0, NT)],
                                             const float (&c)[NT]) {
  int lane = threadIdx.x & 63;
  opaque(lane);
  const int g = lane >> 4, n = lane & 15, cn = sigma(n);
  int bad = 0;
  // the normals: block B of four components on lane B
  if (lane < 32) {
    uint32_t w[4];
    philox_at(a.seed, (uint32_t)row, (uint32_t)lane, (uint32_t)it, make_tag(TAG_LATENT, a.mode), w);
    float z[4];
    box_muller_f32(w[0], w[1], z[0], z[1]);
    box_muller_f32(w[2], w[3], z[2], z[3]);
#pragma unroll
    for (int u = 0; u < 4; u++)
      reinterpret_cast<float*>(&s.v[lane >> 2][u])[lane & 3] = 4 * lane + u < a.K ? z[u] : 0.f;
  }
  float b[NT];
#pragma unroll
  for (int k = 0; k < NT; k++) {
    const int i = 16 * k + cn;
    b[k] = fmaf(alpha, c[k], a.Lmu_rows ? a.Lmu_rows[(size_t)row * 128 + i] : a.Lmu_f[i]);
  }
#pragma unroll
  for (int j = 0; j < NT; j++) {
#pragma unroll
    for (int i = 0; i < NT; i++) {
      if (i > j) continue;
      const f32x4 l = lam[slot(i, j)][lane];
#pragma unroll
      for (int v = 0; v < 4; v++) P[slot(i, j)][v] = fmaf(alpha, P[slot(i, j)][v], l[v]);
    }
  }
  // factorisation, and the forward solve y_k = L_kk^{-1} (b_k - sum_i R_ik^T y_i):
  // y_k in the rows' order (register v = component 4v + g), b's reductions
  // held per row of lanes until their block comes
  f32x4 y[NT];
  float f[NT];
#pragma unroll
  for (int k = 0; k < NT; k++) f[k] = 0.f;
#pragma unroll
  for (int k = 0; k < NT; k++) {
    // (the fences keep the compiler from stretching registers across steps)
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 li = diag_factor(P[slot(k, k)], lane, bad);
    __builtin_amdgcn_sched_barrier(0);
    P[slot(k, k)] = li;
    if (k + 1 < NT) {
      s.t[lane] = li;
      lds_wait();
      f32x4 la;  // as left operand: L_kk^{-1}[component cn][4v + g]
      const float* T = reinterpret_cast<const float*>(s.t);
#pragma unroll
      for (int v = 0; v < 4; v++) la[v] = T[4 * (16 * (cn & 3) + 4 * g + v) + (cn >> 2)];
#pragma unroll
      for (int j = 0; j < NT; j++)
        if (j > k) P[slot(k, j)] = mul_add(la, P[slot(k, j)], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < NT; i++) {
        if (i <= k) continue;
        const f32x4 m = -P[slot(k, i)];
#pragma unroll
        for (int j = 0; j < NT; j++)
          if (j >= i) P[slot(i, j)] = mul_add(m, P[slot(k, j)], P[slot(i, j)]);
      }
    }
    const float t = b[k] - sum_rows(f[k]);
#pragma unroll
    for (int v = 0; v < 4; v++) y[k][v] = sum16(li[v] * t);
#pragma unroll
    for (int j = 0; j < NT; j++) {
      if (j <= k) continue;
#pragma unroll
      for (int v = 0; v < 4; v++) f[j] = fmaf(P[slot(k, j)][v], y[k][v], f[j]);
    }
  }
  // u_k = L_kk^{-T} (y_k + z_k - sum_j>k R_kj u_j), from the last block up; the
  // sums over the lanes of a row taken when their block comes
  lds_wait();
  f32x4 t[NT];
#pragma unroll
  for (int k = 0; k < NT; k++) t[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  double sse = 0.0;
  float ww = 0.f, uc = 0.f;
#pragma unroll
  for (int kk = 0; kk < NT; kk++) {
    const int k = NT - 1 - kk;
    const f32x4 z = s.v[k][g];
    float u = 0.f;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const float x = y[k][v] + z[v];
      ww = n == 0 ? fmaf(x, x, ww) : ww;
      u = fmaf(P[slot(k, k)][v], x - sum16(t[k][v]), u);
    }
    u = sum_rows(u);
#pragma unroll
    for (int i = 0; i < NT; i++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (i < k) t[i][v] = fmaf(P[slot(i, k)][v], u, t[i][v]);
    if (g == 0) {
      a.U[(size_t)row * 128 + 16 * k + cn] = u;
      uc = fmaf(u, c[k], uc);
      if (a.sse_partial) reinterpret_cast<float*>(&s.v[k][cn & 3])[cn >> 2] = u;
    }
  }
  for (int i = 16 * NT + lane; i < 128; i += 64) a.U[(size_t)row * 128 + i] = 0.f;
  if (a.sse_partial) {
    // u^T G u - 2 u c + sum r^2, with u^T G u = (|L^T u|^2 - u Lambda u) / alpha
    lds_wait();
    float q1 = 0.f, q2 = 0.f;  // diagonal and off-diagonal tiles
    for (int j = 0; j < NT; j++) {
      const float uj = reinterpret_cast<const float*>(&s.v[j][cn & 3])[cn >> 2];
      for (int i = 0; i <= j; i++) {
        const f32x4 l = lam[slot(i, j)][lane], ui = s.v[i][g];
        const float x = (l[0] * ui[0] + l[1] * ui[1] + l[2] * ui[2] + l[3] * ui[3]) * uj;
        if (i == j) q1 += x;
        else q2 += x;
      }
    }
    sse = ((double)ww - q1 - 2.0 * q2) / alpha - 2.0 * uc;
    if (lane == 0) sse += a.r2[row];
  }
  lds_wait();
  if (bad && lane == 0) atomicMax(a.fail, row + 1);
  return sse;
}

// work-group sum of the lanes' SSE shares into sse_partial[at]
template <int NO, int NT>
__device__ void write_sse128(const SampleArgs& a, double acc, int at, Shared128<NO, NT>& s) {
  if (!a.sse_partial) return;
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  __syncthreads();
  double* red = reinterpret_cast<double*>(s.lam);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = red[0];
    for (int q = 1; q < kWaves128; q++) t += red[q];
    a.sse_partial[at] = t;
  }
}

// the RHS sums of the wave's blocks over the four rows of lanes
template <int NO>
__device__ __forceinline__ void store_sums(Lds128<NO>& s, float* out, int w, const float (&sums)[2]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const float c = sum_rows(sums[h]);
    if (lane < 16) out[32 * w + 16 * h + sigma(lane)] = c;
  }
}

template <int NO, int NT>
__global__ void __launch_bounds__(64 * kWaves128) k_light128(SampleArgs a, BatchPlan p) {
  __shared__ Shared128<NO, NT> s;
  const Factors<NO> F = make_factors<NO, 128>(a.others);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = *a.iter;
  const float alpha = (float)(*a.alpha);
  load_lambda(a, s);
  double sse = 0.0;
  for (int q = blockIdx.x + gridDim.x * w; q < p.n_pair; q += gridDim.x * kWaves128) {
    const int4 rng = p.pair_rng[q];
    f32x4 P[slot(0, NT)];
    float c[NT];
    gram_row<NO, NT>(a, F, s.wave[w], rng.x, rng.y, P, c);
    sse += finish_row<NO, NT>(a, p.pair_row[q].x, it, alpha, s.lam, s.wave[w], P, c);
  }
  write_sse128(a, sse, blockIdx.x, s);
}

// The same for fewer rows than the chip holds waves: S waves (2, 4 or 8) take a
// share of a row's nonzeros each, and one of them, in turn, finishes the row
// while the others go on to the next.  Their tiles are added through the LDS
// that holds the factors' low parts, NT tiles at a time: each of the S waves adds
// its share of those tiles, in the order of the waves.
template <int NO, int NT>
__global__ void __launch_bounds__(64 * kWaves128) k_light128w(SampleArgs a, BatchPlan p, int S) {
  __shared__ Shared128<NO, NT> s;
  const Factors<NO> F = make_factors<NO, 128>(a.others);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = *a.iter;
  const float alpha = (float)(*a.alpha);
  load_lambda(a, s);
  const int R = kWaves128 / S, u = w % R, part = w / R;  // rows a turn; the wave's row and share
  double sse = 0.0;
  int turn = 0;
  for (int q0 = blockIdx.x; q0 < p.n_pair; q0 += gridDim.x * R, turn++) {
    const int q = q0 + gridDim.x * u;
    const int4 rng = q < p.n_pair ? p.pair_rng[q] : make_int4(0, 0, 0, 0);
    const int share = (rng.y - rng.x + 32 * S - 1) / (32 * S) * 32;
    const int b = min(rng.x + part * share, rng.y);
    f32x4 P[slot(0, NT)];
    float c[NT];
    gram_row<NO, NT>(a, F, s.wave[w], b, min(b + share, rng.y), P, c);
    const int f = turn % S;  // the share whose wave finishes
    if (lane < 16) {
#pragma unroll
      for (int I = 0; I < NT; I++) reinterpret_cast<float*>(s.wave[w].t)[16 * I + lane] = c[I];
    }
#pragma unroll
    for (int t0 = 0; t0 < slot(0, NT); t0 += NT) {
#pragma unroll
      for (int k = 0; k < NT; k++)
        if (t0 + k < slot(0, NT)) s.wave[w].lo[k][lane] = __builtin_bit_cast(uint4, P[t0 + k]);
      __syncthreads();
      for (int k = part; k < NT && t0 + k < slot(0, NT); k += S) {
        f32x4 x = __builtin_bit_cast(f32x4, s.wave[u].lo[k][lane]);
        for (int m = 1; m < S; m++) x += __builtin_bit_cast(f32x4, s.wave[m * R + u].lo[k][lane]);
        s.wave[f * R + u].lo[k][lane] = __builtin_bit_cast(uint4, x);
      }
      if (t0 == 0 && part == f) {
#pragma unroll
        for (int I = 0; I < NT; I++) {
          c[I] = 0.f;
          for (int m = 0; m < S; m++) c[I] += reinterpret_cast<const float*>(s.wave[m * R + u].t)[16 * I + (lane & 15)];
        }
      }
      __syncthreads();
      if (part == f) {
#pragma unroll
        for (int k = 0; k < NT; k++)
          if (t0 + k < slot(0, NT)) P[t0 + k] = __builtin_bit_cast(f32x4, s.wave[w].lo[k][lane]);
      }
    }
    if (part == f && q < p.n_pair)
      sse += finish_row<NO, NT>(a, p.pair_row[q].x, it, alpha, s.lam, s.wave[w], P, c);
  }
  write_sse128(a, sse, blockIdx.x, s);
}

// nb: the component blocks that the finishing kernel reads.  It may be compiled
// for more than K has, so the tiles beyond (zero) are stored too.
template <int NO>
__global__ void __launch_bounds__(kThreads128, 2) k_seg128(SampleArgs a, BatchPlan p, int nb) {
  __shared__ Lds128<NO> s;
  const Factors<NO> F = make_factors<NO, 128>(a.others);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nt = (a.K + 15) / 16;
  Gram128<NO> G(a, F, s, nt);
  for (int sg = blockIdx.x; sg < p.n_seg; sg += gridDim.x) {
    f32x4 acc[10];
    float sums[2];
    G.open(p.seg_beg[sg], p.seg_end[sg]);
    G.start();
    G.run(acc, sums);
    float* out = p.partial + (size_t)sg * kPartial128;
    gram_tiles(w, nb, [&](int t, int i, int j) { *reinterpret_cast<f32x4*>(out + 256 * slot(i, j) + 4 * lane) = acc[t]; });
    store_sums(s, out + 256 * kTiles, w, sums);
    __syncthreads();  // the operand buffers are reused by the next segment
  }
}

template <int NT>
__global__ void __launch_bounds__(64 * kWaves128) k_heavy128(SampleArgs a, BatchPlan p, int sse_slot0) {
  __shared__ Shared128<1, NT> s;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = *a.iter;
  const float alpha = (float)(*a.alpha);
  load_lambda(a, s);
  double sse = 0.0;
  for (int q = blockIdx.x + gridDim.x * w; q < p.n_heavy; q += gridDim.x * kWaves128) {
    // the slot's summed partial (k_seg_sum leaves it in the first segment)
    const float* in = p.partial + (size_t)p.heavy_seg0[q] * kPartial128;
    f32x4 P[slot(0, NT)];
    float c[NT];
#pragma unroll
    for (int t = 0; t < slot(0, NT); t++) P[t] = *reinterpret_cast<const f32x4*>(in + 256 * t + 4 * lane);
#pragma unroll
    for (int I = 0; I < NT; I++) c[I] = in[256 * kTiles + 16 * I + sigma(lane & 15)];
    sse += finish_row<1, NT>(a, p.heavy[q], it, alpha, s.lam, s.wave[w], P, c);
  }
  write_sse128(a, sse, sse_slot0 + blockIdx.x, s);
}

// Waves that share a light row: as many as the rows leave free of the chip's 2048
// (one work-group of eight a CU).  A wave takes 2 to 4 us for 32 nonzeros (the
// gathers of one 16-component block after the other), the finish of a row 40 us.
// Half-sweep in us with 1 | 2 | 4 | 8 waves a row, by rows x nonzeros, K = 128:
//   64 x 100         43 | 45 | 40 | 39
//   64 x 2000       242 | 186 | 116 | 82
//   300 x 200        56 | 55 | 49 | 76
//   300 x 2000      241 | 184 | 122 | 147
//   1000 x 100       48 | 52 | 79 | 139
//   1000 x 1000     158 | 133 | 155 | 209
//   2000 x 1000     227 | 241 | 294 | 411
// (a second round of work-groups, from 257 rows on with a grid of 512: 102 us at
// 300 x 200, 463 at 300 x 2000).
int waves_per_row(const BatchPlan& p) {
  return p.n_light <= k128Grid ? 8 : p.n_light <= 2 * k128Grid ? 4 : p.n_light <= 4 * k128Grid ? 2 : 1;
}

template <int NO, int NT>
void launch128_t(const SampleArgs& a, const BatchPlan& p, hipStream_t s, const SegStreams& seg) {
  const int gl = batched_light_grid(p), gh = batched_heavy_grid(p);
  const bool fork = p.n_seg > 0 && seg.stream;
  if (p.n_seg > 0) {
    const hipStream_t ss = fork ? seg.stream : s;
    if (fork) seg_fork(s, seg);
    hipLaunchKernelGGL((k_seg128<NO>), dim3(batched_seg_grid(p)), dim3(kThreads128), 0, ss, a, p, NT);
    launch_seg_sum<kPartial128>(p, ss);
    if (gh > 0) hipLaunchKernelGGL((k_heavy128<NT>), dim3(gh), dim3(64 * kWaves128), 0, ss, a, p, gl);
    if (fork) seg_record_join(seg);
  }
  const int S = waves_per_row(p);
  if (gl > 0 && S > 1) hipLaunchKernelGGL((k_light128w<NO, NT>), dim3(gl), dim3(64 * kWaves128), 0, s, a, p, S);
  else if (gl > 0) hipLaunchKernelGGL((k_light128<NO, NT>), dim3(gl), dim3(64 * kWaves128), 0, s, a, p);
  if (fork) seg_wait_join(s, seg);
}

// one kernel per number of component blocks for matrices and 3-mode tensors
// (at K = 70 five of eight blocks are 15 of 36 tiles); larger tensors take all
// eight
template <int NO>
void launch128_k(const SampleArgs& a, const BatchPlan& p, hipStream_t s, const SegStreams& seg) {
  if constexpr (NO <= 2) {
    switch ((a.K + 15) / 16) {
      case 5: return launch128_t<NO, 5>(a, p, s, seg);
      case 6: return launch128_t<NO, 6>(a, p, s, seg);
      case 7: return launch128_t<NO, 7>(a, p, s, seg);
      default: break;
    }
  }
  launch128_t<NO, 8>(a, p, s, seg);
}

}  // namespace

// A work-group's waves take rows gridDim.x apart, so that few rows spread over
// the CUs first
int batched128_light_grid(const BatchPlan& p) {
  return std::min(p.n_pair, p.light_cap > 0 ? p.light_cap : batched_light_default(p));
}
int batched128_heavy_grid(const BatchPlan& p) {
  return std::min(p.n_heavy, p.heavy_cap > 0 ? p.heavy_cap : batched_heavy_default(p));
}

void launch_sample_batched128(const SampleArgs& a, const BatchPlan& p, hipStream_t s, const SegStreams& seg) {
  switch (a.rows.nother) {
    case 1: return launch128_k<1>(a, p, s, seg);
    case 2: return launch128_k<2>(a, p, s, seg);
    case 3: return launch128_k<3>(a, p, s, seg);
    case 4: return launch128_k<4>(a, p, s, seg);
    default: break;
  }
}

}  // namespace mgpu
