// A norm and the dense layer behind it in one launch, for up to 128 rows: 16 rows per
// workgroup, normed once for many columns.
#include "common.h"
#include "gemm_tiles.h"
#include "norm_dense.h"

namespace t5d {

// The workgroups of a launch, and which row tile of which columns each takes.  All row tiles of
// the same columns go to one XCD, whose L2 has the weights then, and columns to the XCDs in turn
// where that gives none more workgroups than its 32 CUs.  For 3, 5, 6 and 7 row tiles it may
// give some 33 to 36 of up to 256, and these a second round (steps of 112 rows, width 1024, 599
// us, two kernels 582; of 80 rows 508 and 516): then each takes an eighth of all in a row
// (567 and 496).
struct Work {
  int blocks, per_xcd, part;  // part: 65536 / row tiles, rounded up (exact for 8 and 2^12)
  Work(int N, int nt, int m_parts) {
    const int groups = (N / 16 + 2 * nt - 1) / (2 * nt), columns = (groups + 7) / 8;
    per_xcd = columns * m_parts > 32 ? (groups * m_parts + 7) / 8 : 0;
    blocks = 8 * (per_xcd ? per_xcd : columns * m_parts);
    part = (65536 + m_parts - 1) / m_parts;
  }
};

// 512 threads own 16 rows and 2 NT column tiles.  Each of the 8 wavefronts norms two whole
// rows, without a barrier; they meet the matrix cores through LDS.  For the products wavefront
// (half, part) = (w / 4, w % 4) takes NT of the column tiles and every fourth pair of k-tiles
// (KQ at most), so the sums have the order of gemm_mfma_kernel.  All of a wavefront's weights
// are requested behind its rows and arrive while these are normed.
// What bounds it: the chain launch (2 us), rows, sums over them, products, sum over the
// wavefronts, and what a CU takes in of weights that come from memory: 64 KB of them (NT = 1
// at 1024 inputs) 1.2 us; from its XCD's L2 it takes 150 to 220 bytes per ns (128 KB in 0.6
// to 0.9 us).  So columns are spread over as many CUs as there are, and no further: each
// workgroup norms its rows anew.  us, weights from memory:
//   norm in norm_gemm_kernel / here       rows 16       32            64            128
//     768 x 2304                     3.90          4.34 / 3.95   5.31 / 4.45   6.61 / 5.30
//     768 x 4096 gated               4.38          4.91 / 4.35   5.84 / 4.80   7.28
//     1024 x 3072                    4.69          5.19 / 4.57   6.46 / 5.30   7.97 / 6.92
//     1024 x 5632 gated              5.89 / 5.52   7.30 / 6.40   9.02 / 7.80  12.08
//     512 x 5632 gated               4.09          4.88 / 4.10   5.92 / 5.10   7.21
//     1024 x 5632 gated, int8        5.58 / 5.10   6.94 / 6.18   8.98 / 7.73  12.50
//   float32 stream, two kernels / here
//     512 x 3328                     6.20 / 5.04   6.50 / 5.12   7.04 / 5.51   7.98 / 6.70
//     768 x 4096 gated               6.55 / 6.00   6.87 / 6.16   7.79 / 6.76   9.52 / 8.18
//     1024 x 3328                    6.63 / 6.45   7.07 / 6.72   8.35 / 7.58  10.12 / 9.70
//     1024 x 5632 gated              8.06 / 7.31   8.69 / 8.28  10.37 / 9.82  12.91 / 18.6
// A row in the lanes' own groups of 4 columns, its norm through LDS and another barrier, was
// slower than these pieces, each half a wavefront reading what the other does too (64 x 1024 x
// 5632 8.46 / 7.96, 64 x 768 x 2304 4.65 / 4.55), and gave sums another order.  What stands in
// front of the first load counts: a second division there, or gridDim, 0.3 to 0.5 us.
// Tried and slower: 16 wavefronts (64 x 1024 x 5632 8.85), 4 (8.94), 32 rows per workgroup
// with K over 8 wavefronts (8.67, 64 x 768 x 4096 6.70 instead of 5.36).
template <typename Args, int NT, int KQ, typename WT>
__global__ void __launch_bounds__(512)
norm_dense_kernel(Args g, Work work) {
  constexpr bool kStream = IsStream<Args>::value, kLatent = IsLatent<Args>::value;
  constexpr bool kPlain = !kStream && !kLatent;
  constexpr int LD = 256 * KQ, HS = LD + 8;  // row stride of the normed rows
  constexpr int TB = WeightTile<WT>::kTileBytes, TN = 32 * NT;
  __shared__ __align__(16) bf16_t s_h[16 * HS];
  __shared__ float red[8][NT * 4][64];
  __shared__ __align__(16) float s_norm[kStream ? 2 : 1][kPlain ? 4 : LD];
  T5D_GATE_READ(g.gate);
  if constexpr (kLatent) {
    if ((int)blockIdx.x >= g.dense_blocks) {  // a cached latent per wavefront
      const int m = 8 * (blockIdx.x - g.dense_blocks) + (threadIdx.x >> 6);
      T5D_GATE_TEST();
      if (m >= g.M) return;
      const int at = 8 * (threadIdx.x & 63), have = (g.kv_d + 15) & ~15;
      const bf16_t* row = g.kv + (size_t)m * g.lda;
      bf16_t* dst = g.ring + ((size_t)g.seq_slot[g.tok_seq[m]] * g.ring_len +
                              g.tok_pos[m] % g.ring_len) * g.kv_pad;
      float ss = 0.f;
      for (int c = at; c < have; c += 512) {
        float f[8];
        unpack16(latent_piece(row, c, have), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
      }
      const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)g.kv_d + g.eps);
      for (int c = at; c < g.kv_pad; c += 512)
        *reinterpret_cast<uint4*>(dst + c) =
            latent_normed(latent_piece(row, c, have), inv, g.kv_norm + c);
      return;
    }
  }
  const int xcd = blockIdx.x & 7, slot = (blockIdx.x >> 3) + xcd * work.per_xcd;
  const int q = slot * work.part >> 16, m_part = slot - q * g.m_parts;
  const int n_group = work.per_xcd ? q : q * 8 + xcd;
  const int n_tiles_total = g.N >> 4, nt0 = n_group * 2 * NT;
  if (nt0 >= n_tiles_total) return;
  const int m0 = m_part * 16;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave >> 2, part = wave & 3;
  const int K = g.K, KT = K >> 5, n_pairs = KT >> 1;

  // The norms' vectors (4 columns of one or of both per thread), two rows per wavefront in
  // groups of 4 columns, the weights: in the order in which they are used.  (Plain rows: in
  // the pieces that norm_gemm_kernel adds up, a row in lanes % 32 / 16, twice; lane l norms
  // half l / 32 of each.)
  constexpr int PV = (LD / 4 + 511) / 512;
  float4 vec[PV], vec_y[kStream ? PV : 1];
  const int d = columns_of_norm(g);
#pragma unroll
  for (int v = 0; !kPlain && v < PV; ++v) {
    const int c = 4 * (threadIdx.x + 512 * v);
    if constexpr (kStream) {
      vec_y[v] = g.y_norm != nullptr ? norm_column(g.y_norm, c, d)
                                     : make_float4(1.f, 1.f, 1.f, 1.f);
      vec[v] = norm_column(g.norm, c, d);
    } else if constexpr (kLatent) {
      vec[v] = norm_column(g.norm, c, d);
    }
  }
  constexpr int KP8 = (KQ + 1) / 2;  // groups of 8 columns per lane
  uint4 x8[kLatent ? 2 : 1][KP8];
  const int have = kLatent ? (d_of_norm(g) + 15) & ~15 : 0;
  float4 x[kStream ? 2 : 1][KQ];
  uint2 y[2][KQ];
  const bool add = has_branch(g);
  const int p_row = 2 * wave + (lane >> 4 & 1), p_half = lane >> 5;
  const int p_at = 64 * (lane >> 2 & 3) + 8 * (lane & 3);
  uint4 xp[kPlain ? KQ : 1][2], sp[kPlain ? KQ : 1];
  if constexpr (kPlain) {
    const bf16_t* from = g.A + (size_t)min(m0 + p_row, g.M - 1) * K + p_at;
#pragma unroll
    for (int j = 0; j < KQ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        xp[j][h] = p_at + 256 * j < K
                       ? *reinterpret_cast<const uint4*>(from + 256 * j + 32 * h)
                       : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < KQ; ++j)
      sp[j] = p_at + 256 * j < K ? *reinterpret_cast<const uint4*>(g.norm_scale + p_at +
                                                                   256 * j + 32 * p_half)
                                 : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; !kPlain && r < 2; ++r) {
    // (past the end: the last row, not stored)
    const size_t row = (size_t)min(m0 + 2 * wave + r, g.M - 1) * row_stride(g);
    if constexpr (kLatent) {
#pragma unroll
      for (int q = 0; q < KP8; ++q)
        x8[r][q] = latent_piece(g.A + row, 8 * lane + 512 * q, have);
    }
#pragma unroll
    for (int q = 0; !kLatent && q < KQ; ++q) {
      const int c = 4 * lane + 256 * q;
      const bool on = c < K;
      y[r][q] = make_uint2(0, 0);
      if constexpr (kStream) {
        x[r][q] = on ? *reinterpret_cast<const float4*>(g.x + row + c)
                     : make_float4(0.f, 0.f, 0.f, 0.f);
        if (on && add) y[r][q] = *reinterpret_cast<const uint2*>(g.y + row + c);
      }
    }
  }
  typename WeightTile<WT>::Raw w[KQ][2][NT];
#pragma unroll
  for (int j = 0; j < KQ; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int nn = 0; nn < NT; ++nn)
        w[j][h][nn] = WeightTile<WT>::load(
            reinterpret_cast<const char*>(g.W) +
                ((size_t)min(nt0 + half * NT + nn, n_tiles_total - 1) * KT +
                 2 * min(part + 4 * j, n_pairs - 1) + h) * TB,
            lane);
  T5D_GATE_TEST();
  if constexpr (!kPlain) {
#pragma unroll
    for (int v = 0; v < PV; ++v) {
      const int c = 4 * (threadIdx.x + 512 * v);
      if (c < LD) {
        *reinterpret_cast<float4*>(&s_norm[0][c]) = vec[v];
        if constexpr (kStream) *reinterpret_cast<float4*>(&s_norm[1][c]) = vec_y[v];
      }
    }
    // (what is requested may come later: no wait for it at the barriers)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }

  if constexpr (kStream) {
    // as stream_norm_kernel, whose 4 wavefronts hold columns 256 w + 1024 v of a row: one
    // sum per w
    constexpr int SW = KQ < 4 ? KQ : 4;
    const auto row_sum = [&](const float (&s)[4]) { return (s[0] + s[1]) + (s[2] + s[3]); };
    float inv[2] = {1.f, 1.f};
    if (add) {
      const bool normed = g.y_norm != nullptr;
      if (normed) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = 0; q < KQ; ++q) {
            const float y0 = bf16lo_to_f32(y[r][q].x), y1 = bf16hi_to_f32(y[r][q].x);
            const float y2 = bf16lo_to_f32(y[r][q].y), y3 = bf16hi_to_f32(y[r][q].y);
            float& a = s[q & 3];
            a = fmaf(y0, y0, a); a = fmaf(y1, y1, a);
            a = fmaf(y2, y2, a); a = fmaf(y3, y3, a);
          }
#pragma unroll
          for (int i = 0; i < SW; ++i) s[i] = wave_sum(s[i]);
          inv[r] = 1.0f / sqrtf(row_sum(s) / (float)d + g.eps);
        }
      }
#pragma unroll
      for (int q = 0; q < KQ; ++q) {
        const int c = 4 * lane + 256 * q;
        const float4 wy = *reinterpret_cast<const float4*>(&s_norm[kStream ? 1 : 0][c]);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          x[r][q].x += bf16lo_to_f32(y[r][q].x) * inv[r] * wy.x;
          x[r][q].y += bf16hi_to_f32(y[r][q].x) * inv[r] * wy.y;
          x[r][q].z += bf16lo_to_f32(y[r][q].y) * inv[r] * wy.z;
          x[r][q].w += bf16hi_to_f32(y[r][q].y) * inv[r] * wy.w;
          const int m = m0 + 2 * wave + r;
          if (n_group == 0 && m < g.M && c < K)
            *reinterpret_cast<float4*>(g.x_out + (size_t)m * K + c) = x[r][q];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < KQ; ++q) {
        float& a = s[q & 3];
        a = fmaf(x[r][q].x, x[r][q].x, a); a = fmaf(x[r][q].y, x[r][q].y, a);
        a = fmaf(x[r][q].z, x[r][q].z, a); a = fmaf(x[r][q].w, x[r][q].w, a);
      }
#pragma unroll
      for (int i = 0; i < SW; ++i) s[i] = wave_sum(s[i]);
      inv[r] = 1.0f / sqrtf(row_sum(s) / (float)d + g.eps);
    }
#pragma unroll
    for (int q = 0; q < KQ; ++q) {
      const int c = 4 * lane + 256 * q;
      const float4 wx = *reinterpret_cast<const float4*>(&s_norm[0][c]);
#pragma unroll
      for (int r = 0; r < 2; ++r)
        *reinterpret_cast<uint2*>(s_h + (2 * wave + r) * HS + c) = make_uint2(
            pack_bf16x2(x[r][q].x * inv[r] * wx.x, x[r][q].y * inv[r] * wx.y),
            pack_bf16x2(x[r][q].z * inv[r] * wx.z, x[r][q].w * inv[r] * wx.w));
    }
  } else if constexpr (kLatent) {  // (summed as latent_append_kernel does)
    float inv[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      float ss = 0.f;
#pragma unroll
      for (int q = 0; q < KP8; ++q) {
        float f[8];
        unpack16(x8[r][q], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
      }
      inv[r] = 1.0f / sqrtf(wave_sum(ss) / (float)d_of_norm(g) + g.eps);
    }
#pragma unroll
    for (int q = 0; q < KP8; ++q) {
      const int c = 8 * lane + 512 * q;
      if (KQ % 2 != 0 && c >= LD) break;
#pragma unroll
      for (int r = 0; r < 2; ++r)
        *reinterpret_cast<uint4*>(s_h + (2 * wave + r) * HS + c) =
            latent_normed(x8[r][q], inv[r], &s_norm[0][c]);
    }
  } else {
    // (summed as norm_gemm_kernel does, so that a row has the same bits in both: its wavefronts
    // w are lanes % 16 / 4 here)
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < KQ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float f[8];
        unpack16(xp[j][h], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
      }
    ss += dpp_move<kDppXor1>(ss);
    ss += dpp_move<kDppXor2>(ss);
    ss += lane_xor8(ss);
    ss += lane_xor4(ss);
    const float inv = 1.0f / sqrtf(ss / (float)K + g.eps);
#pragma unroll
    for (int j = 0; j < KQ; ++j) {
      float xf[8], sf[8];
      unpack16(p_half ? xp[j][1] : xp[j][0], xf);
      unpack16(sp[j], sf);
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t n = pack_bf16x2(xf[2 * e] * inv, xf[2 * e + 1] * inv);
        o[e] = pack_bf16x2(bf16lo_to_f32(n) * sf[2 * e], bf16hi_to_f32(n) * sf[2 * e + 1]);
      }
      *reinterpret_cast<uint4*>(s_h + p_row * HS + p_at + 256 * j + 32 * p_half) =
          make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  f32x4_v acc[NT];
#pragma unroll
  for (int nn = 0; nn < NT; ++nn) acc[nn] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  const bf16_t* a_from = s_h + (lane & 15) * HS + 8 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < KQ; ++j) {
    const int pair = part + 4 * j;
    if (pair >= n_pairs) break;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      Frag a;
      a.u = *reinterpret_cast<const uint4*>(a_from + 64 * pair + 32 * h);
#pragma unroll
      for (int nn = 0; nn < NT; ++nn)
        acc[nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a.v, WeightTile<WT>::frag(w[j][h][nn]).v, acc[nn], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][t * 4 + i][lane] = acc[t][i];
  __syncthreads();
  const bool pair = gated(g);
  const auto tile_sum = [&](int ml, int nl) -> float {
    const int l = (ml >> 2) * 16 + (nl & 15), t = nl >> 4;
    const int b = t >= NT ? 4 : 0, idx = (t - (t >= NT ? NT : 0)) * 4 + (ml & 3);
    return (red[b][idx][l] + red[b + 2][idx][l]) + (red[b + 1][idx][l] + red[b + 3][idx][l]);
  };
#pragma unroll
  for (int p = 0; p < NT; ++p) {
    const int e = threadIdx.x + 512 * p;
    const int ml = e / TN, nl = e % TN, m = m0 + ml, n = nt0 * 16 + nl;
    if (m >= g.M || n >= stored_columns(g) || (pair && (nl & 8))) continue;
    float v = tile_sum(ml, nl), vg = pair ? tile_sum(ml, nl + 8) : 0.f;
    if (g.scales != nullptr) {
      v *= g.scales[n];
      if (pair) vg *= g.scales[n + 8];
    }
    store_result(g, m, n, v, vg, 0.f);
  }
}

// Column tiles per half of a workgroup: as few as leave every workgroup a CU of its own (the
// second round costs more than the wider workgroup: 64 x 1024 x 5632 8.16 us with 3, 8.82
// with 2); 0 where even `most` do not.
static int tiles_per_half(int M, int N, int most) {
  const int m_parts = (M + 15) / 16, tiles = N / 16;
  for (int nt = 1; nt <= most; ++nt)
    if ((tiles + 2 * nt - 1) / (2 * nt) * m_parts <= 256) return nt;
  return 0;
}

template <typename Args, typename WT>
static void launch(int nt, Args g, hipStream_t s) {
  g.m_parts = (g.M + 15) / 16;
  const Work work(g.N, nt, g.m_parts);
  const dim3 grid(work.blocks), block(512);
#define T5D_ND_K(NT_, KQ_)                                                             \
  hipLaunchKernelGGL((norm_dense_kernel<Args, NT_, KQ_, WT>), grid, block, 0, s, g, work)
#define T5D_ND(NT_)                          \
  do {                                       \
    if (g.K <= 512) T5D_ND_K(NT_, 2);        \
    else if (g.K <= 768) T5D_ND_K(NT_, 3);   \
    else T5D_ND_K(NT_, 4);                   \
  } while (0)
  if (nt == 1) T5D_ND(1);
  else if (nt == 2) T5D_ND(2);
  else if (nt == 3) T5D_ND(3);
  else if constexpr (IsStream<Args>::value) T5D_ND(4);
  else T5D_ND_K(4, 2);  // (launch_norm_dense: 4 tiles up to 512 inputs)
#undef T5D_ND
#undef T5D_ND_K
}

// Where norm_gemm_kernel has more than one workgroup per CU (512 inputs: more than two; 48 x
// 512 x 2304 3.75 us there, 3.87 here; 16 x 1024 x 4096 5.12 / 5.15), and the columns fit
// 256 workgroups: beyond 512 inputs with up to 3 tiles (4 there: 80 x 768 x 5632 7.55 / 7.80,
// 128 x 1024 x 4096 8.44 / 8.87; 128 x 512 x 4096 5.83 / 5.49).
bool launch_norm_dense(int w_dtype, const GemmArgs& g, hipStream_t s) {
  if (g.K > 1024) return false;
  const int nt = tiles_per_half(g.M, g.N, g.K <= 512 ? 4 : 3);
  if (nt == 0 || g.N / 16 * ((g.M + 15) / 16) <= (g.K <= 512 ? 512 : 256)) return false;
  if (w_dtype == T5D_I8) launch<GemmArgs, int8_t>(nt, g, s);
  else launch<GemmArgs, bf16_t>(nt, g, s);
  return true;
}

// Up to 128 rows whose columns fit 256 workgroups of four column tiles (two halves of two).
// Steps of 8 layers, 4 of them with a cache of their own, us with two launches / so, rows 1,
// 8, 64, 128: 6 heads of 128 (width 768) 405 / 387, 497 / 480, 646 / 624, 821 / 799; 8 heads
// 458 / 435, 562 / 539, 756 / 732, 963 / 936; 16 heads 649 / 627, 863 / 837, 1414 / 1382,
// 1722 / 1687.
bool launch_latent_dense(LatentDenseArgs g, hipStream_t s) {
  if (g.M > 128 || g.K > 1024 || g.K % 64 != 0) return false;
  const int nt = tiles_per_half(g.M, g.N, 2);
  if (nt == 0) return false;
  g.m_parts = (g.M + 15) / 16;
  const Work work(g.N, nt, g.m_parts);
  g.dense_blocks = work.blocks;
  const dim3 grid(g.dense_blocks + (g.kv != nullptr ? (g.M + 7) / 8 : 0)), block(512);
#define T5D_LD_K(NT_, KQ_)                                                               \
  hipLaunchKernelGGL((norm_dense_kernel<LatentDenseArgs, NT_, KQ_, bf16_t>), grid, block, \
                     0, s, g, work)
#define T5D_LD(NT_)                        \
  do {                                     \
    if (g.K <= 512) T5D_LD_K(NT_, 2);      \
    else if (g.K <= 768) T5D_LD_K(NT_, 3); \
    else T5D_LD_K(NT_, 4);                 \
  } while (0)
  if (nt == 1) T5D_LD(1);
  else T5D_LD(2);
#undef T5D_LD
#undef T5D_LD_K
  return true;
}

}  // namespace t5d

using namespace t5d;

extern "C" int t5d_stream_rows_dense_rows(int dtype, int ld) {
  return dtype == T5D_BF16 && ld > 0 && ld % 64 == 0 && ld <= 1024 ? 128 : 0;
}

// Where the columns fit 256 workgroups of at most 8 column tiles (80 x 1024 x 8192 13.8 us as
// two kernels, 18 here) and, beyond 768 inputs, take more than one tile of each: for fewer both
// are the same within a few percent (16 x 1024 x 2304 6.37 / 6.43, 33 x 1024 x 1024 6.39 / 6.43,
// 16 x 1024 x 3328 6.63 / 6.45; 24 x 1024 x 2304 6.87 / 6.55, 16 x 1024 x 5632 8.06 / 7.31).
// There four tiles of each half also want more than 192 workgroups (33 x 896 x 8192, 192, 10.25 /
// 10.94; 64 x 896 x 8192, 256, 11.4 / 11.2; three tiles pay with 177: steps with a gated layer of
// 33 x 1024 x 5632 378 / 372), and for 64 and 128 inputs three and four tiles do not pay (33 x
// 64 x 8192 5.53 / 5.80, 80 x 128 x 4608 5.78 / 5.97).
extern "C" int t5d_stream_rows_dense_pays(int M, int ld, int N) {
  const int nt = tiles_per_half(M, N, 4), m_parts = (M + 15) / 16, tiles = N / 16;
  if (nt == 0 || ld <= 128) return nt > 0 && nt < 3;
  return ld <= 768 || (tiles * m_parts > 256 &&
                       (nt < 4 || (tiles + 2 * nt - 1) / (2 * nt) * m_parts > 192));
}

extern "C" int t5d_stream_rows_dense(void* stream, const void* y, const float* y_norm,
                                     const float* x, float* x_out, const float* norm, int d,
                                     float eps, const void* W, int out_dtype, void* C,
                                     int ldc, int n_store, int M, int ld, int N,
                                     int epilogue, float glu_limit, float glu_alpha,
                                     float glu_add) {
  StreamDenseArgs g;
  const int rc = stream_dense_args("t5d_stream_rows_dense", &g,
                                   t5d_stream_rows_dense_rows(T5D_BF16, ld), y, y_norm, x,
                                   x_out, norm, d, eps, W, out_dtype, C, ldc, n_store, M, ld,
                                   N, epilogue, glu_limit, glu_alpha, glu_add);
  if (rc != T5D_OK) return rc;
  const int nt = tiles_per_half(M, N, 4);
  launch<StreamDenseArgs, bf16_t>(nt ? nt : 4, g, as_stream(stream));
  T5D_CHECK_LAUNCH("t5d_stream_rows_dense");
  return T5D_OK;
}
