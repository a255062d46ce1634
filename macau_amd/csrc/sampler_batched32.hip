// sampler_batched32.hip -- nnz-bucketed per-row sampler with a split-BF16 MFMA
// Gram for K in (16, 32], four rows per wave.
//
// Same mathematics as sample_latent_blas (latentprior.cpp:361-385) and
// sample_latent_tensor (latentprior.cpp:118-161): per row
//   P = Lambda + alpha G,  G = sum_e c_e c_e^T,  b = alpha sum_e c_e r_e + Lambda mu_n,
//   u = L^{-T}(L^{-1} b + z),  P = L L^T.
//
// Work decomposition of one half-sweep (BatchPlan, built on the host):
//   * rows with more than 2048 nonzeros are split into 2048-nnz segments;
//     k_seg32 computes each segment's partial Gram and RHS (one wave per
//     segment), k_seg_sum adds each row's partials in segment order (one
//     thread per partial entry), and k_heavy32 finishes four rows per wave;
//   * the other rows, sorted by nnz (descending), are taken in fours by
//     k_light32 (similar nnz keeps the four busy alike).
// Layout: the 16 x 16 tiles (0,0), (0,1), (1,1) of the matrix in the accumulators
// of v_mfma_*_16x16x*: lane (g, n) = (l / 16, l % 16) has in register v the entry
// (4g + v, n).
// Gram (QuadStream): the wave takes one row's nonzeros 32 at a time, lane
// (g, n) components n and n + 16 of nonzeros 8g .. 8g + 7, which is the operand
// layout of v_mfma_f32_16x16x32_bf16.  Every value is split into hi = bf16(x) and
// lo = bf16(x - hi), and a tile accumulates Hi Hi^T + Hi Lo^T + Lo Hi^T + Lo Lo^T
// in FP32.  Without Lo Lo^T the diagonal loses a positive bias of ~5e-6 |x|^2
// per product, which rows of few nonzeros against a weak prior direction turn
// into row errors near 1e-4.  Up to kThreeParts light rows there is a middle part
// too (24 bits; the split is then nearly all of the error).  The RHS accumulates in FP32
// on the vector ALU.
// Finish (finish_quad): row q of the four is taken over by lanes 16q .. 16q + 15,
// which hold rows n and n + 16 of its matrix: everything that all lanes of a
// row do alike (4 x 4 blocks, broadcasts) is done for four rows at once.  Two rows
// a wave with 32 x 32 tiles took 538 us at 138000 rows x 133 nonzeros and 275 at
// 27000 x 680 (17.7 MB of factors, read through the last-level cache), these
// take 353 and 230.  Bound by vector instructions (the split, the RHS, the
// finish: about half of the time at two waves a SIMD) and the gathers' latency;
// three waves a SIMD spill 21 registers and take 364 and 239.
// Adaptive noise: for the last mode the train SSE of the new samples is
// accumulated as u^T G u - 2 u^T c + sum r^2 per row, with
// u^T G u = (|L^{-1} b + z|^2 - u^T Lambda u) / alpha (since L^T u = L^{-1} b + z),
// so no separate pass over the nonzeros is needed.
#include <stdexcept>

#include "batched.h"

namespace mgpu {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int NT = 2;                                 // 16-component blocks
constexpr int kTiles32 = 3;                           // their tiles
constexpr int kThreeParts = 12000;                    // light rows up to which factors are split into three parts
constexpr int kPartial32 = kTiles32 * 256 + NT * 64;  // floats per segment partial: tiles and RHS sums per lane

__device__ __forceinline__ void lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// lane k's value on every lane of its row of 16
template <int k>
__device__ __forceinline__ float bcast16(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + k, 0xf, 0xf, true));  // row_newbcast
}
// sum over the 16 lanes of a row of lanes
template <int CTRL>
__device__ __forceinline__ float ror_add(float x) {
  return x + __builtin_bit_cast(
                 float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum16(float x) { return ror_add<0x121>(ror_add<0x122>(ror_add<0x124>(ror_add<0x128>(x)))); }

__device__ __forceinline__ void swap32(float& x, float& y) {  // x's lanes 32-63 <-> y's lanes 0-31
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& x, float& y) {  // x's odd rows of 16 lanes <-> y's even rows
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}
// x[k] of lanes 16q + n  ->  x[q] of lanes 16k + n
__device__ __forceinline__ void transpose4(float (&x)[4]) {
  swap32(x[0], x[2]);
  swap32(x[1], x[3]);
  swap16(x[0], x[1]);
  swap16(x[2], x[3]);
}
// the sum over the rows of lanes of x[q], on row q of lanes
__device__ __forceinline__ float sum_rows4(float x0, float x1, float x2, float x3) {
  swap32(x0, x2);
  swap32(x1, x3);
  float a = x0 + x2, b = x1 + x3;
  swap16(a, b);
  return a + b;
}
__device__ __forceinline__ int sel4(int g, int4 x) {
  const int lo = g & 1 ? x.y : x.x, hi = g & 1 ? x.w : x.z;
  return g & 2 ? hi : lo;
}

// ---------------------------------------------------------------------------
// Gram stream over the nonzeros of ROWS rows, in blocks of 64 (two chunks of
// 32; a block never spans two rows, a row has at least one).  Per block:
//   1. each lane loads one nonzero's indices and residual (coalesced), two
//      blocks ahead;
//   2. the block is staged in LDS, and each lane reads, per chunk, the 8 indices
//      of its row of lanes with two 16-byte broadcast reads and gathers its
//      components of those 8 factor columns with bounds-checked buffer loads
//      (index -1 = padding reads as 0), one block ahead: a chunk's values are
//      requested as soon as the previous block's are split;
//   3. the chunks go through the split-BF16 MFMA.
// ---------------------------------------------------------------------------
template <int NO>
struct QuadBlk {
  alignas(16) int ix[2][NO][64];  // double buffered
  alignas(16) float r[2][64];
};

template <int NO, int ROWS, int PARTS>
struct QuadStream {
  const SampleArgs& a;
  const Factors<NO>& F;
  QuadBlk<NO>& L;
  int beg[ROWS], end[ROWS];
  int lane, g, n;
  int e1, end1, q1;  // the next block: its start, its row's end and its row
  int buf = 0;
  BlkReg<NO> nxt;    // its indices
  float v[2][NT][8];

  __device__ __forceinline__ QuadStream(const SampleArgs& a_, const Factors<NO>& F_, QuadBlk<NO>& L_,
                                        const int4 (&r)[(ROWS + 1) / 2])
      : a(a_), F(F_), L(L_) {
    lane = threadIdx.x & 63;
    g = lane >> 4;
    n = lane & 15;
    rows(r);
  }
  __device__ __forceinline__ void rows(const int4 (&r)[(ROWS + 1) / 2]) {
#pragma unroll
    for (int q = 0; q < ROWS; q++) {
      beg[q] = q & 1 ? r[q / 2].z : r[q / 2].x;
      end[q] = q & 1 ? r[q / 2].w : r[q / 2].y;
    }
  }
  static __device__ __forceinline__ void pick(const int (&x)[ROWS], int q, int& out) {
    out = 0;
#pragma unroll
    for (int u = 0; u < ROWS; u++) out = q == u ? x[u] : out;
  }
  __device__ __forceinline__ void advance() {
    if (e1 + 64 < end1) {
      e1 += 64;
    } else {
      q1++;
      pick(beg, q1, e1);
      pick(end, q1, end1);
    }
  }
  // the first two blocks' indices and residuals, issued ahead of time by a
  // caller and handed to run()
  __device__ __forceinline__ void first_blocks(BlkReg<NO>& b0, BlkReg<NO>& b1) {
    e1 = beg[0];
    end1 = end[0];
    q1 = 0;
    load_blk<NO, 64>(a, e1, end1, lane, b0);
    advance();
    load_blk<NO, 64>(a, e1, end1, lane, b1);
  }
  __device__ __forceinline__ void stage(const BlkReg<NO>& b) {
#pragma unroll
    for (int t = 0; t < NO; t++) L.ix[buf][t][lane] = b.ix[t];
    L.r[buf][lane] = b.r;
    lds_order();
  }
  template <int c>
  __device__ __forceinline__ void gather() {
    i32x4 ix[NO][2];
#pragma unroll
    for (int t = 0; t < NO; t++) {
      ix[t][0] = *reinterpret_cast<const i32x4*>(&L.ix[buf][t][32 * c + 8 * g]);
      ix[t][1] = *reinterpret_cast<const i32x4*>(&L.ix[buf][t][32 * c + 8 * g + 4]);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      int at[NO];
#pragma unroll
      for (int t = 0; t < NO; t++) at[t] = factor_at<32>(ix[t][i >> 2][i & 3], n);
#pragma unroll
      for (int h = 0; h < NT; h++) {
        float x = ld_at(F.rs[0], at[0], 16 * h);
#pragma unroll
        for (int t = 1; t < NO; t++) x *= ld_at(F.rs[t], at[t], 16 * h);
        v[c][h][i] = x;
      }
    }
  }
  // chunk c of the current block (in v and buffer buf ^ 1) into T and cs, and
  // the gathers of the next block's chunk c (staged in buffer buf)
  template <int c>
  __device__ __forceinline__ void chunk(f32x4 (&T)[kTiles32], float (&cs)[NT]) {
    const f32x4 r0 = *reinterpret_cast<const f32x4*>(&L.r[buf ^ 1][32 * c + 8 * g]);
    const f32x4 r1 = *reinterpret_cast<const f32x4*>(&L.r[buf ^ 1][32 * c + 8 * g + 4]);
    bf16x8 x[NT][3];  // hi, (mid,) lo
#pragma unroll
    for (int h = 0; h < NT; h++) {
#pragma unroll
      for (int i = 0; i < 4; i++) cs[h] = fmaf(v[c][h][i], r0[i], cs[h]);
#pragma unroll
      for (int i = 0; i < 4; i++) cs[h] = fmaf(v[c][h][4 + i], r1[i], cs[h]);
      if (PARTS == 3) split8(v[c][h], x[h][0], x[h][1], x[h][2]);
      else split8(v[c][h], x[h][0], x[h][1]);
    }
    gather<c>();
#pragma unroll
    for (int t = 0; t < kTiles32; t++)
#pragma unroll
      for (int i = 0; i < PARTS; i++)
#pragma unroll
        for (int j = 0; j < PARTS; j++)
          if (i + j < 3) T[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t == 2][i], x[t != 0][j], T[t], 0, 0, 0);
  }
  template <int TR>
  __device__ __forceinline__ void run(const BlkReg<NO>& b0, const BlkReg<NO>& b1, f32x4 (&T)[TR][kTiles32],
                                      float (&cs)[TR][NT]) {
    lds_order();
    stage(b0);
    gather<0>();
    gather<1>();
    nxt = b1;
#pragma unroll
    for (int q = 0; q < ROWS; q++) {
#pragma unroll
      for (int t = 0; t < kTiles32; t++) T[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < NT; h++) cs[q][h] = 0.f;
      int e = beg[q];
      do {
        buf ^= 1;
        stage(nxt);
        advance();
        load_blk<NO, 64>(a, e1, end1, lane, nxt);
        chunk<0>(T[q], cs[q]);
        if (e + 32 < end[q]) chunk<1>(T[q], cs[q]);
        else gather<1>();
        lds_order();
        e += 64;
      } while (e < end[q]);
    }
  }
};

// L in 4-column blocks s (columns 4s .. 4s + 3 of rows 4s and below, 4 floats
// each, blocks 4 floats further apart than their sizes) and rows kQuadRow floats
// apart: the back solve's reads of one row of L, 16 lanes for each of four
// matrices, hit every bank twice.
__device__ __forceinline__ constexpr int l_off(int s) { return s * (64 * NT + 4) - 8 * s * (s - 1); }
template <int NO>
struct QuadLds {
  static constexpr int kRow = 624;
  alignas(16) float L[4 * kRow];
  union {
    QuadBlk<NO> blk;       // of the Gram stream
    f32x4 W[4][16 * NT];   // the current block columns of -P, per row
  };
  f32x4 y[4][4 * NT];    // forward solution and reciprocal pivots, later the samples
  f32x4 rp[4][4 * NT];
  f32x4 z[4][4 * NT];    // the normals
};

// The 4-column step k0 = 4 s of the factorisation, with the forward solve.
template <int s, typename Lds>
struct QuadStep {
  static constexpr int k0 = 4 * s, h0 = s / 4, gs = s % 4;
  static __device__ __forceinline__ void run(f32x4 (&T)[4][kTiles32], float (&b)[NT], bool probe, float (&x)[3][NT],
                                             float (&sq)[3], bool& bad, Lds& S, int K) {
    if (k0 >= K) return;  // uniform
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    // row of lanes gs holds the block's columns (rows, by symmetry) of every
    // matrix; lane (q, n) reads rows n, n + 16 and the diagonal block of matrix q
    if (g == gs) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (h0 == 0) {
          S.W[q][n] = T[q][0];
          S.W[q][16 + n] = T[q][1];
        } else {
          S.W[q][16 + n] = T[q][2];
        }
      }
    }
    lds_order();
    f32x4 w[NT], d[4];
#pragma unroll
    for (int t = 0; t < 4; t++) d[t] = S.W[g][k0 + t];
#pragma unroll
    for (int h = h0; h < NT; h++) w[h] = S.W[g][16 * h + n];
    lds_order();
    // L_D = chol(-d)
    const float a00 = -d[0][0];
    bool bp = !(a00 > 0.f);
    const float r0 = __builtin_amdgcn_rsqf(bp ? 1.f : a00);
    const float l10 = -d[1][0] * r0, l20 = -d[2][0] * r0, l30 = -d[3][0] * r0;
    const float a11 = -d[1][1] - l10 * l10;
    bp = bp || !(a11 > 0.f);
    const float r1 = __builtin_amdgcn_rsqf(a11 > 0.f ? a11 : 1.f);
    const float l21 = (-d[2][1] - l20 * l10) * r1, l31 = (-d[3][1] - l30 * l10) * r1;
    const float a22 = -d[2][2] - l20 * l20 - l21 * l21;
    bp = bp || !(a22 > 0.f);
    const float r2 = __builtin_amdgcn_rsqf(a22 > 0.f ? a22 : 1.f);
    const float l32 = (-d[3][2] - l30 * l20 - l31 * l21) * r2;
    const float a33 = -d[3][3] - l30 * l30 - l31 * l31 - l32 * l32;
    bp = bp || !(a33 > 0.f);
    const float r3 = __builtin_amdgcn_rsqf(a33 > 0.f ? a33 : 1.f);
    bad = bad || bp;
    // the lane's rows of the block's columns of L, and their elimination from
    // the RHS.  A lane inside the block gets its row of L_D; one above it gets
    // values that nothing reads.
    float p[NT][4];
#pragma unroll
    for (int h = h0; h < NT; h++) {
      p[h][0] = -w[h][0] * r0;
      p[h][1] = (-w[h][1] - p[h][0] * l10) * r1;
      p[h][2] = (-w[h][2] - p[h][0] * l20 - p[h][1] * l21) * r2;
      p[h][3] = (-w[h][3] - p[h][0] * l30 - p[h][1] * l31 - p[h][2] * l32) * r3;
      if (16 * h + n >= k0)
        *reinterpret_cast<f32x4*>(&S.L[g * Lds::kRow + l_off(s) + 4 * (16 * h + n - k0)]) =
            f32x4{p[h][0], p[h][1], p[h][2], p[h][3]};
    }
    auto forward = [&](float (&c)[NT]) {
      f32x4 y;
      y[0] = bcast16<k0 % 16>(c[h0]) * r0;
      y[1] = (bcast16<k0 % 16 + 1>(c[h0]) - l10 * y[0]) * r1;
      y[2] = (bcast16<k0 % 16 + 2>(c[h0]) - l20 * y[0] - l21 * y[1]) * r2;
      y[3] = (bcast16<k0 % 16 + 3>(c[h0]) - l30 * y[0] - l31 * y[1] - l32 * y[2]) * r3;
#pragma unroll
      for (int h = h0; h < NT; h++)
#pragma unroll
        for (int t = 0; t < 4; t++) c[h] = fmaf(-p[h][t], y[t], c[h]);
      return y;
    };
    const f32x4 y = forward(b);
    if (n == 0) {
      S.y[g][s] = y;
      S.rp[g][s] = f32x4{r0, r1, r2, r3};
    }
    if (probe) {
#pragma unroll
      for (int u = 0; u < 3; u++) {
        const f32x4 t = forward(x[u]);
        sq[u] += t[0] * t[0] + t[1] * t[1] + t[2] * t[2] + t[3] * t[3];
      }
    }
    // -P += p p^T: row k of lanes passes column k of its matrix
    if (s + 1 < 4 * NT) {
#pragma unroll
      for (int h = h0; h < NT; h++) transpose4(p[h]);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (gs < 3) {
          T[q][h0 == 0 ? 0 : 2] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(p[h0][q], p[h0][q], T[q][h0 == 0 ? 0 : 2], 0, 0, 0);
          if (h0 == 0)
            T[q][1] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(p[0][q], p[1][q], T[q][1], 0, 0, 0);
        }
        if (h0 == 0)
          T[q][2] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(p[1][q], p[1][q], T[q][2], 0, 0, 0);
      }
    }
  }
};

// Row j of the back solve L^T u = w, from the last: x = w inv on lane j % 16 of
// each row of lanes is u_j; w of the components above loses L[j][.] u_j.
template <int j>
__device__ __forceinline__ void back_row(float (&w)[NT], const float (&inv)[NT], const float* const (&Lp)[NT], int n) {
  const float x = bcast16<j % 16>(w[j / 16] * inv[j / 16]);
  if (j / 16 == 1) w[0] = fmaf(-Lp[0][4 * j], x, w[0]);
  const float t = fmaf(-Lp[j / 16][4 * j], x, w[j / 16]);
  w[j / 16] = n < j % 16 ? t : w[j / 16];
}

// Finish four rows whose Gram tiles are in T and whose RHS sums over the
// lane's nonzeros in cs (row < 0: none).  Returns this lane's SSE share.
//
// P = Lambda + alpha G stays in the tiles, negated, for the factorisation in
// 4-column blocks (QuadStep): the block's columns go through LDS to the lanes
// of their matrix, which factor the 4 x 4 diagonal block (redundantly) and form
// their rows of L; the rank-4 update of a tile is one v_mfma_f32_16x16x4_f32 on
// those, transposed between rows of lanes by four swaps for all four matrices.
// With refinement on, three probe vectors x (the row's normals z, all ones,
// alternating signs) are forward-solved beside the RHS, giving |L^{-1} x|^2 =
// x^T P^{-1} x for the condition estimate (probe_estimate).
template <typename Lds>
__device__ __forceinline__ float finish_quad(const SampleArgs& a, int4 rows, int4 nnz,
                                             f32x4 (&T)[4][kTiles32], const float (&cs)[4][NT], int it, float alpha,
                                             Lds& S) {
  int lane = threadIdx.x & 63;
  opaque(lane);
  const int g = lane >> 4, n = lane & 15;
  const int row = sel4(g, rows);
  const bool active = row >= 0;
  if (lane < 32) {
    // four normals a lane
    const int q = lane / (4 * NT), B = lane % (4 * NT);
    const int zr = sel4(q, rows);
    uint32_t w[4];
    philox_at(a.seed, (uint32_t)(zr < 0 ? 0 : zr), (uint32_t)B, (uint32_t)it, make_tag(TAG_LATENT, a.mode), w);
    float z[4];
    box_muller_f32(w[0], w[1], z[0], z[1]);
    box_muller_f32(w[2], w[3], z[2], z[3]);
#pragma unroll
    for (int u = 0; u < 4; u++) z[u] = 4 * B + u < a.K ? z[u] : 0.f;
    S.z[q][B] = f32x4{z[0], z[1], z[2], z[3]};
  }
#pragma unroll
  for (int t = 0; t < kTiles32; t++) {
    const f32x4 l = *reinterpret_cast<const f32x4*>(a.Lambda_f + (n + (t > 0 ? 16 : 0)) * 32 + 4 * g + (t == 2 ? 16 : 0));
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) T[q][t][v] = -fmaf(alpha, T[q][t][v], l[v]);
  }
  float c[NT], b[NT];
#pragma unroll
  for (int h = 0; h < NT; h++) {
    c[h] = sum_rows4(cs[0][h], cs[1][h], cs[2][h], cs[3][h]);
    const int i = 16 * h + n;
    b[h] = fmaf(alpha, c[h], a.Lmu_rows ? (active ? a.Lmu_rows[(size_t)row * 32 + i] : 0.f) : a.Lmu_f[i]);
  }
  lds_order();
  // condition probes (refinement only): L^{-1} D^{1/2} x for x = z, ones,
  // alternating signs, D = diag(P)
  const int mnnz = a.refine.min_nnz;
  const bool probe = a.refine.count != nullptr &&
                     max(max(nnz.x, nnz.y), max(nnz.z, nnz.w)) >= mnnz;
  float x[3][NT], sq[3] = {0.f, 0.f, 0.f}, zz = 0.f;
  if (probe) {
    // the diagonals: lane (n / 4, n) has entry n of a tile in register n % 4
#pragma unroll
    for (int h = 0; h < NT; h++) {
      if (g == n >> 2) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const f32x4 t = T[q][h == 0 ? 0 : 2];
          const float lo = n & 1 ? t[1] : t[0], hi = n & 1 ? t[3] : t[2];
          reinterpret_cast<float*>(S.W[q])[16 * h + n] = n & 2 ? hi : lo;
        }
      }
    }
    lds_order();
#pragma unroll
    for (int h = 0; h < NT; h++) {
      const int i = 16 * h + n;
      const float sd = sqrtf(-reinterpret_cast<const float*>(S.W[g])[i]);
      const float z = reinterpret_cast<const float*>(S.z[g])[i];
      zz += z * z;
      x[0][h] = z * sd;
      x[1][h] = i < a.K ? sd : 0.f;
      x[2][h] = i < a.K ? ((i & 1) ? -sd : sd) : 0.f;
    }
    lds_order();
    zz = sum16(zz);
  }
  bool bad = false;
  QuadStep<0, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<1, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<2, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<3, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<4, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<5, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<6, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  QuadStep<7, Lds>::run(T, b, probe, x, sq, bad, S, a.K);
  if (bad && active && n == 0) atomicMax(a.fail, row + 1);
  lds_order();
  float w[NT], ws[NT], inv[NT];
  const float* Lp[NT];
#pragma unroll
  for (int h = 0; h < NT; h++) {
    const int i = 16 * h + n, s = i >> 2;
    const bool in = i < a.K;  // steps past K are not taken
    w[h] = in ? reinterpret_cast<const float*>(S.y[g])[i] + reinterpret_cast<const float*>(S.z[g])[i] : 0.f;
    ws[h] = w[h];
    inv[h] = in ? reinterpret_cast<const float*>(S.rp[g])[i] : 0.f;
    Lp[h] = S.L + g * Lds::kRow + l_off(s) - 16 * s + (n & 3);
  }
#define BACK4(s)                     \
  if (4 * (s) < a.K) {               \
    back_row<4 * (s) + 3>(w, inv, Lp, n); \
    back_row<4 * (s) + 2>(w, inv, Lp, n); \
    back_row<4 * (s) + 1>(w, inv, Lp, n); \
    back_row<4 * (s)>(w, inv, Lp, n);     \
  }
  BACK4(7) BACK4(6) BACK4(5) BACK4(4) BACK4(3) BACK4(2) BACK4(1) BACK4(0)
#undef BACK4
  float u[NT];
#pragma unroll
  for (int h = 0; h < NT; h++) {
    u[h] = w[h] * inv[h];
    if (active) a.U[(size_t)row * 32 + 16 * h + n] = u[h];
  }
  const int my_nnz = sel4(g, nnz);
  if (probe) {
    const float est = probe_value(a.K, sq[0], sq[1], sq[2], zz);
    const RefineQueue& Q = a.refine;
    const bool flag = active && my_nnz >= Q.min_nnz && est > Q.thresh;
    int slot = -1;
    if (flag && n == 0) {
      slot = atomicAdd(Q.count, 1);
      if (slot < Q.cap) Q.row[slot] = row;
    }
    slot = __shfl(slot, g * 16, 64);
    if (flag && slot >= 0 && slot < Q.cap) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int i = 16 * h + n;
        float* dst = Q.L + (size_t)slot * 1024 + (size_t)i * 32;
#pragma unroll
        for (int s = 0; s < 8; s++) {
          f32x4 t = {0.f, 0.f, 0.f, 0.f};
          if (4 * s <= i && 4 * s < a.K) {
            t = *reinterpret_cast<const f32x4*>(&S.L[g * Lds::kRow + l_off(s) + 4 * (i - 4 * s)]);
#pragma unroll
            for (int k = 1; k < 4; k++) t[k] = 4 * s + k <= i ? t[k] : 0.f;
          }
          if (i >= (a.K + 3) / 4 * 4) {  // steps past K: the identity
#pragma unroll
            for (int k = 0; k < 4; k++) t[k] = 4 * s + k == i ? 1.f : 0.f;
          }
          *reinterpret_cast<f32x4*>(dst + 4 * s) = t;
        }
      }
    }
  }
  if (!a.sse_partial) return 0.f;
  // train SSE share of this lane: (w^2 - u (Lambda u)) / alpha - 2 u c (+ sum r^2)
  float* us = reinterpret_cast<float*>(S.y[g]);
#pragma unroll
  for (int h = 0; h < NT; h++) us[16 * h + n] = u[h];
  lds_order();
  float lu[NT];
#pragma unroll
  for (int h = 0; h < NT; h++) {
    const float* Lrow = a.Lambda_f + (16 * h + n) * 32;
    lu[h] = 0.f;
#pragma unroll
    for (int q = 0; q < 4 * NT; q++) {
      const f32x4 l = *reinterpret_cast<const f32x4*>(Lrow + 4 * q), x4 = S.y[g][q];
      lu[h] += l[0] * x4[0] + l[1] * x4[1] + l[2] * x4[2] + l[3] * x4[3];
    }
  }
  lds_order();
  float t = 0.f;
  if (active) {
#pragma unroll
    for (int h = 0; h < NT; h++) t += (ws[h] * ws[h] - u[h] * lu[h]) / alpha - 2.f * u[h] * c[h];
    if (n == 0) t += a.r2[row];
  }
  return t;
}

// Wave q takes the pairs 2q, 2q + 1 of the plan, then those G waves further
// (G = grid).  Row ids and ranges come from the plan in one load a pair, and the
// next rows' ranges and their first two index blocks are loaded while the
// current ones are finished.
template <int NO, int PARTS>
__global__ void __launch_bounds__(64, 2) k_light32(SampleArgs a, BatchPlan p) {
  __shared__ QuadLds<NO> S;
  const Factors<NO> F = make_factors<NO, 32>(a.others);
  const int it = *a.iter;
  const float alpha = (float)(*a.alpha);
  double sse = 0.0;
  const int n = (p.n_pair + 1) / 2;
  int4 rng[2];
  int2 rows[2];
  auto plan = [&](int q) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const bool in = 2 * q + u < p.n_pair;
      rng[u] = in ? p.pair_rng[2 * q + u] : make_int4(0, 0, 0, 0);
      rows[u] = in ? p.pair_row[2 * q + u] : make_int2(-1, -1);
    }
  };
  int q = blockIdx.x;
  BlkReg<NO> b0, b1;
  if (q < n) plan(q);
  QuadStream<NO, 4, PARTS> gs(a, F, S.blk, rng);
  if (q < n) gs.first_blocks(b0, b1);
  while (q < n) {
    f32x4 T[4][kTiles32];
    float cs[4][NT];
    gs.run(b0, b1, T, cs);
    const int4 rw = make_int4(rows[0].x, rows[0].y, rows[1].x, rows[1].y);
    const int4 nz = make_int4(rng[0].y - rng[0].x, rng[0].w - rng[0].z, rng[1].y - rng[1].x, rng[1].w - rng[1].z);
    q += gridDim.x;
    if (q < n) {
      plan(q);
      gs.rows(rng);
      gs.first_blocks(b0, b1);
    }
    sse += (double)finish_quad(a, rw, nz, T, cs, it, alpha, S);
  }
  write_sse(a, sse, blockIdx.x);
}

// The same for fewer rows than fill the chip with waves: a work-group of four
// waves takes R = 4, 2 or 1 rows, 4 / R waves the Gram of one each, and its waves
// in turn finish the rows while the others go on to the next.
template <int NO>
struct WideLds {
  QuadLds<NO> S;
  QuadBlk<NO> blk[4];
  f32x4 T[2][4][kTiles32][64];
  float cs[2][4][NT][64];
  double sse[4];
};
template <int NO, int R>
__global__ void __launch_bounds__(256, NO == 1 ? 3 : 2) k_light32w(SampleArgs a, BatchPlan p) {
  __shared__ WideLds<NO> S;
  const Factors<NO> F = make_factors<NO, 32>(a.others);
  const int it = *a.iter;
  const float alpha = (float)(*a.alpha);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double sse = 0.0;
  int turn = 0;
  // row i of the plan: its range, and its id
  auto range = [&](int i) {
    const int4 r = i < p.n_light ? p.pair_rng[i >> 1] : make_int4(0, 0, 0, 0);
    return i & 1 ? make_int2(r.z, r.w) : make_int2(r.x, r.y);
  };
  for (int i0 = R * blockIdx.x; i0 < p.n_light; i0 += R * gridDim.x, turn++) {
    const int buf = turn & 1;
    {
      const int2 r = range(i0 + w % R);
      const int share = R == 4 ? r.y - r.x : ((r.y - r.x + 256 / R - 1) / (256 / R)) * 64;
      const int4 mine[1] = {make_int4(min(r.x + (w / R) * share, r.y), min(r.x + (w / R + 1) * share, r.y), 0, 0)};
      f32x4 T[1][kTiles32];
      float cs[1][NT];
      BlkReg<NO> b0, b1;
      QuadStream<NO, 1, 3> gs(a, F, S.blk[w], mine);
      gs.first_blocks(b0, b1);
      gs.run(b0, b1, T, cs);
#pragma unroll
      for (int t = 0; t < kTiles32; t++) S.T[buf][w][t][lane] = T[0][t];
#pragma unroll
      for (int h = 0; h < NT; h++) S.cs[buf][w][h][lane] = cs[0][h];
    }
    __syncthreads();
    if (w == (turn & 3)) {
      f32x4 T[4][kTiles32];
      float cs[4][NT];
      int id[4], nz[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
#pragma unroll
        for (int t = 0; t < kTiles32; t++) {
          T[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (u < R) T[u][t] = S.T[buf][u][t][lane];
#pragma unroll
          for (int k = u + R; u < R && k < 4; k += R) T[u][t] += S.T[buf][k][t][lane];
        }
#pragma unroll
        for (int h = 0; h < NT; h++) {
          cs[u][h] = u < R ? S.cs[buf][u][h][lane] : 0.f;
#pragma unroll
          for (int k = u + R; u < R && k < 4; k += R) cs[u][h] += S.cs[buf][k][h][lane];
        }
        id[u] = -1;
        nz[u] = 0;
        if (u < R && i0 + u < p.n_light) {
          const int2 r = range(i0 + u), pr = p.pair_row[(i0 + u) >> 1];
          id[u] = (i0 + u) & 1 ? pr.y : pr.x;
          nz[u] = r.y - r.x;
        }
      }
      sse += (double)finish_quad(a, make_int4(id[0], id[1], id[2], id[3]), make_int4(nz[0], nz[1], nz[2], nz[3]), T,
                                     cs, it, alpha, S.S);
    }
  }
  if (!a.sse_partial) return;
  for (int off = 32; off > 0; off >>= 1) sse += __shfl_down(sse, off, 64);
  if (lane == 0) S.sse[w] = sse;
  __syncthreads();
  if (threadIdx.x == 0) a.sse_partial[blockIdx.x] = ((S.sse[0] + S.sse[1]) + S.sse[2]) + S.sse[3];
}

template <int NO>
__global__ void __launch_bounds__(64) k_seg32(SampleArgs a, BatchPlan p) {
  __shared__ QuadBlk<NO> blk;
  const Factors<NO> F = make_factors<NO, 32>(a.others);
  const int lane = threadIdx.x;
  for (int sg = blockIdx.x; sg < p.n_seg; sg += gridDim.x) {
    const int4 r[1] = {make_int4(p.seg_beg[sg], p.seg_end[sg], 0, 0)};
    f32x4 T[1][kTiles32];
    float cs[1][NT];
    BlkReg<NO> b0, b1;
    QuadStream<NO, 1, 2> gs(a, F, blk, r);
    gs.first_blocks(b0, b1);
    gs.run(b0, b1, T, cs);
    float* out = p.partial + (size_t)sg * kPartial32;
#pragma unroll
    for (int t = 0; t < kTiles32; t++) *reinterpret_cast<f32x4*>(out + 256 * t + 4 * lane) = T[0][t];
#pragma unroll
    for (int h = 0; h < NT; h++) out[kTiles32 * 256 + 64 * h + lane] = cs[0][h];
  }
}

// four heavy rows per wave, from their summed partials (k_seg_sum leaves them
// in each row's first segment)
__global__ void __launch_bounds__(64) k_heavy32(SampleArgs a, BatchPlan p, int sse_slot0) {
  __shared__ QuadLds<1> S;
  const int lane = threadIdx.x;
  const int it = *a.iter;
  const float alpha = (float)(*a.alpha);
  double sse = 0.0;
  for (int q = blockIdx.x; 4 * q < p.n_heavy; q += gridDim.x) {
    f32x4 T[4][kTiles32];
    float cs[4][NT];
    int r[4], z[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const bool in = 4 * q + u < p.n_heavy;
      r[u] = in ? p.heavy[4 * q + u] : -1;
      z[u] = in ? p.seg_len : 0;
      const float* src = p.partial + (size_t)p.heavy_seg0[in ? 4 * q + u : 4 * q] * kPartial32;
#pragma unroll
      for (int t = 0; t < kTiles32; t++) {
        T[u][t] = *reinterpret_cast<const f32x4*>(src + 256 * t + 4 * lane);
        if (!in) T[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int h = 0; h < NT; h++) cs[u][h] = in ? src[kTiles32 * 256 + 64 * h + lane] : 0.f;
    }
    sse += (double)finish_quad(a, make_int4(r[0], r[1], r[2], r[3]), make_int4(z[0], z[1], z[2], z[3]), T, cs, it,
                                   alpha, S);
  }
  write_sse(a, sse, sse_slot0 + blockIdx.x);
}

// Light rows per work-group of four waves (0: four a wave, k_light32).  Half-sweep
// in us with 1 | 2 | 4 rows | four a wave, by rows x nonzeros a row, K = 32, three
// parts a factor:
//   300 x 512        19 | 21 | 25 | 43
//   1500 x 256       32 | 23 | 24 | 31
//   3000 x 1         45 | 28 | 19 | 19
//   5000 x 128       69 | 44 | 31 | 30
//   5000 x 500       97 | 74 | 58 | 66   (27000 factor columns)
//   8000 x 1        102 | 58 | 36 | 23
//   8000 x 500      145 | 104 | 83 | 73
//   8000, up to 2048 (power law)  105 | 102 | 148   (2 | 4 rows | four a wave)
// Few rows: the time is that of the longest row's gathers, one block of 64 after
// the other, and of one finish.  Many: the finish of four rows at once by every
// wave counts, and a work-group's three idle waves in it do not pay, unless the
// longest rows, four of them one after the other on a wave, take longer still.
static int rows_per_group(const BatchPlan& p) {
  if (p.n_light <= 512) return 1;
  if (p.n_light <= 1024) return 2;
  if (p.n_light <= 3000) return 4;
  return p.n_light <= kThreeParts && p.light_max > p.n_light / 12 ? 4 : 0;
}

// Four rows a wave: without a cap of the plan's, 16384 waves, which take the
// rows in 2 strides at 138000 x 32 (5% less time than 8192 waves, 30% less than
// 3072: fewer waves with more rows each end less evenly).
int batched32_light_default(const BatchPlan& p) {
  return rows_per_group(p) ? kDefaultLightCap : 2 * kDefaultLightCap;
}
int batched32_light_grid(const BatchPlan& p) {
  const int r = rows_per_group(p), n = r ? (p.n_light + r - 1) / r : (p.n_pair + 1) / 2;
  const int cap = p.light_cap > 0 ? p.light_cap : batched32_light_default(p);
  return n < cap ? n : cap;
}
int batched32_heavy_grid(const BatchPlan& p) {
  const int n = (p.n_heavy + 3) / 4;
  const int cap = p.heavy_cap > 0 ? p.heavy_cap : kDefaultHeavyCap;
  return n < cap ? n : cap;
}

template <int NO>
static void launch_batched32_t(const SampleArgs& a, const BatchPlan& p, hipStream_t s, const SegStreams& seg) {
  const int gl = batched32_light_grid(p), gh = batched32_heavy_grid(p);
  const bool fork = p.n_seg > 0 && seg.stream;
  if (p.n_seg > 0) {
    const hipStream_t ss = fork ? seg.stream : s;
    if (fork) seg_fork(s, seg);
    const int gs = batched_seg_grid(p);
    hipLaunchKernelGGL((k_seg32<NO>), dim3(gs), dim3(64), 0, ss, a, p);
    launch_seg_sum<kPartial32>(p, ss);
    // the heavy rows depend only on their segments: finished on the segment
    // stream too, beside the light rows
    if (gh > 0) hipLaunchKernelGGL(k_heavy32, dim3(gh), dim3(64), 0, ss, a, p, gl);
    if (fork) seg_record_join(seg);
  }
  if (gl > 0) {
    switch (rows_per_group(p)) {
      case 1: hipLaunchKernelGGL((k_light32w<NO, 1>), dim3(gl), dim3(256), 0, s, a, p); break;
      case 2: hipLaunchKernelGGL((k_light32w<NO, 2>), dim3(gl), dim3(256), 0, s, a, p); break;
      case 4: hipLaunchKernelGGL((k_light32w<NO, 4>), dim3(gl), dim3(256), 0, s, a, p); break;
      default:
        if (p.n_light <= kThreeParts) hipLaunchKernelGGL((k_light32<NO, 3>), dim3(gl), dim3(64), 0, s, a, p);
        else hipLaunchKernelGGL((k_light32<NO, 2>), dim3(gl), dim3(64), 0, s, a, p);
    }
  }
  if (fork) seg_wait_join(s, seg);
  launch_refine(a, s);
}

void launch_sample_batched32(const SampleArgs& a, const BatchPlan& p, hipStream_t s, const SegStreams& seg) {
  switch (a.rows.nother) {
    case 1: return launch_batched32_t<1>(a, p, s, seg);
    case 2: return launch_batched32_t<2>(a, p, s, seg);
    case 3: return launch_batched32_t<3>(a, p, s, seg);
    case 4: return launch_batched32_t<4>(a, p, s, seg);
    default: break;
  }
}

}  // namespace mgpu
