// Dense layers over many rows (the encoder side: M = batch x encoder length).
//
// Unlike the decode-step GEMMs these are compute-bound.  Two kernels:
// rows_gemm_direct_kernel, further down, and for K = 32 and operands beyond its reach
// rows_gemm_kernel.  There a workgroup (4
// wavefronts, 2 x 2) owns a 256 x 128 output tile, each wavefront a 128 x 64
// sub-tile = 8 x 4 MFMA tiles (v_mfma_f32_16x16x32_bf16).  Per k-tile of 32 the
// workgroup needs 16 activation fragments (16 rows x 64 bytes each) and 8
// packed weight tiles, 1 KB apiece in MFMA operand layout; every wavefront
// fetches 6 of them from memory, parks them in LDS exactly as loaded (lane l
// at byte 16 l: conflict-free both ways), and after one barrier reads the 12
// it multiplies.  Global loads for k + 1 are in flight while k is multiplied;
// two LDS buffers, one barrier per k-tile.  Sharing through LDS cuts the
// operand traffic per matrix instruction to 3/8 of what loading every
// operand per wavefront costs, which is what bounds this shape.
// A packed weight tile has the same lane layout as either MFMA operand, so the
// product can be formed as C (activations as A) or as C^T (weights as A); C^T
// leaves every lane with 4 consecutive output COLUMNS of one row, C with 4
// consecutive ROWS of one column — whichever makes the 8-byte stores
// contiguous in the requested output layout.
#include "common.h"
#include "gemm_tiles.h"

namespace t5d {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_r;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_r;

union FragR {
  uint4 u;
  bf16x8_r v;
};

__device__ __forceinline__ uint32_t i8x2_to_bf16x2(int a, int b) {
  // int8 values are exactly representable in bfloat16.
  return (__float_as_uint((float)a) >> 16) |
         (__float_as_uint((float)b) & 0xFFFF0000u);
}

// A packed weight tile as loaded (`Raw`) and widened to bfloat16 (`frag`).
template <typename WT> struct RowsWeightTile;
template <> struct RowsWeightTile<bf16_t> {
  static constexpr int kTileBytes = 1024;
  typedef uint4 Raw;
  __device__ static __forceinline__ Raw load(const char* tile, int lane) {
    return reinterpret_cast<const uint4*>(tile)[lane];
  }
  __device__ static __forceinline__ uint4 frag(const Raw& r) { return r; }
};
template <> struct RowsWeightTile<int8_t> {
  static constexpr int kTileBytes = 512;
  typedef uint2 Raw;
  __device__ static __forceinline__ Raw load(const char* tile, int lane) {
    return reinterpret_cast<const uint2*>(tile)[lane];
  }
  __device__ static __forceinline__ uint4 frag(const Raw& q) {
    uint4 f;
    f.x = i8x2_to_bf16x2((int8_t)(q.x), (int8_t)(q.x >> 8));
    f.y = i8x2_to_bf16x2((int8_t)(q.x >> 16), (int8_t)(q.x >> 24));
    f.z = i8x2_to_bf16x2((int8_t)(q.y), (int8_t)(q.y >> 8));
    f.w = i8x2_to_bf16x2((int8_t)(q.y >> 16), (int8_t)(q.y >> 24));
    return f;
  }
};

struct RowsGemmArgs {
  const bf16_t* A;         // [M, K]
  const char* W;           // packed tiles [N/16][K/32]
  const float* scales;     // [N] for int8 weights, else null
  const bf16_t* residual;  // [M, N] row-major, or null
  bf16_t* C;
  int M, K, N;
  int epilogue;            // T5D_EPI_*
  int layout;              // T5D_OUT_*
  int E, Ep, H;            // heads layouts: m = b * E + e, n = h * 64 + d
  const int32_t* at;       // value layout: b << 12 | e of every 4 rows instead, or null
  int lda;                 // row stride of A
  float* C32;              // float32 output rows instead of C (rows layout, no
  int ldc, n_store;        // epilogue): row stride, columns stored of the N
  float glu_limit, glu_alpha, glu_add;  // T5D_EPI_CLAMPED_GLU
  const int32_t* gate;     // optional device-side enable flag (rows_gemm_direct_kernel)
  GroupTiles grp;          // GROUPED kernels only, with the next
  int n_tiles;
  // NORM kernels (see rows_gemm_direct_kernel)
  const float* squares_in;   // [parts][M] of A's rows before they were scaled
  int parts;                 // of 64 columns each
  float norm_d, eps;         // columns of such a row
  const bf16_t* next_scale;  // [N]
  bf16_t* scaled;            // [M, N]
  float* squares_out;        // [N / 64, rounded up][M]
  // rows_gemm_pair_kernel: the second layer
  const char* W2;
  const float* scales2;
  bf16_t* C2;
  int N2;
};

__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
  uint2 p;
  p.x = pack_bf16x2(a, b);
  p.y = pack_bf16x2(c, d);
  return p;
}

constexpr int kRowsBM = 256, kRowsBN = 128;  // workgroup tile
constexpr int kRowsMT = 8, kRowsNT = 4;        // MFMA tiles per wavefront

// What a wavefront does with its finished accumulator tiles (m0: its first
// row, nt0: its first 16-column tile) when the product was formed as C, for
// the value layout:
template <int MT, int NT>
__device__ __forceinline__ void rows_epilogue_values(
    const RowsGemmArgs& g, const f32x4_r (&acc)[MT][NT], int m0,
    int nt0, int n_tiles, int l16, int gq, const float* inv = nullptr) {
  // acc[mt][nt][i]: row m = m0 + 16 mt + 4 gq + i, column n = 16 (nt0 + nt) + l16
  // (values layout [B, H, Ep / 32, 64, 32]: 4 consecutive positions per store)
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + 16 * mt + 4 * gq;
    if (m >= g.M) continue;
    int b, e;
    if (g.at) {
      const int p = g.at[m >> 2];
      b = p >> 12;
      e = p & 4095;
    } else {
      b = m / g.E;
      e = m - b * g.E;
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt0 + nt >= n_tiles) continue;
      const int n = 16 * (nt0 + nt) + l16;
      float s = g.scales ? g.scales[n] : 1.f;
      float4 f = make_float4(s, s, s, s);
      if (inv) {
        f = *reinterpret_cast<const float4*>(inv + 16 * mt + 4 * gq);
        f.x *= s; f.y *= s; f.z *= s; f.w *= s;
      }
      const int hh = n >> 6, d = n & 63;
      const size_t o =
          ((((size_t)b * g.H + hh) * (g.Ep >> 5) + (e >> 5)) * 64 + d) * 32 +
          (e & 31);
      *reinterpret_cast<uint2*>(g.C + o) =
          pack4(acc[mt][nt][0] * f.x, acc[mt][nt][1] * f.y, acc[mt][nt][2] * f.z,
                acc[mt][nt][3] * f.w);
    }
  }
}

// ... and when it was formed as C^T, with the stores made whole: a lane holds
// 4 consecutive columns of one row, so storing from the accumulators would
// write 16 rows x 8..32 bytes per instruction.  Each
// wavefront instead parks one 16-row slice at a time in a private piece of
// LDS (rounded to bfloat16, rows padded by 16 bytes) and reads it back with 4
// or 8 lanes per row, 16 bytes per lane: every store instruction then writes
// whole 64-byte (gated) or 128-byte rows, and the residual is read the same
// way.  LDS operations of one wavefront complete in order, so the slices
// follow one another through the same piece without a wait in between; the
// empty asm statements keep the compiler from moving one lane's read above
// another lane's write (to it they are accesses of unrelated addresses).
// DENSE: one of the epilogues of t5d_dense instead: 1 = T5D_EPI_CLAMPED_GLU (first
// column of a pair: gate, second: up), 2 = float32 rows.
// NORM: 1 = results are multiplied by shared[row]; 2 = with the residual added, a row's
// squares go to shared[16-column tile of the workgroup][row], and scaled, it is stored a
// second time.
template <int NT> constexpr int kRowsStageStride = NT == 2 ? 80 : 144;
template <int NT> constexpr int kRowsStageBytes = 16 * kRowsStageStride<NT>;
template <int DENSE, bool SCALED, int MT, int NT, int NORM = 0>
__device__ __forceinline__ void rows_epilogue_staged(
    const RowsGemmArgs& g, const f32x4_r (&acc)[MT][NT], int m0, int nt0,
    int n_tiles, int lane, char* stage, float* shared = nullptr, int wave = 0) {
  static_assert(NT >= 2 && NT <= 4, "a wavefront's slice: 32 to 64 columns");
  const int l16 = lane & 15, gq = lane >> 4;
  // int8 weights: the scale of each of this lane's 4 columns
  float4 sc[NT];
  if constexpr (SCALED) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      sc[nt] = (g.scales && nt0 + nt < n_tiles)
                   ? *reinterpret_cast<const float4*>(g.scales +
                                                      16 * (nt0 + nt) + 4 * gq)
                   : make_float4(1.f, 1.f, 1.f, 1.f);
  }
  float inv[MT];
  if constexpr (NORM == 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) inv[mt] = shared[16 * mt + l16];
  }
  const auto value = [&](int mt, int nt, int i) {
    float v = acc[mt][nt][i];
    if constexpr (SCALED) v *= reinterpret_cast<const float*>(&sc[nt])[i];
    if constexpr (NORM == 1) v *= inv[mt];
    return v;
  };
  if constexpr (DENSE == 2) {
    // A lane holds 4 consecutive columns of one row, a store of them 16 rows of 64 bytes:
    // half lines.  Neighbouring tiles trade, so that a store has whole lines, 8 rows of 128
    // bytes.  us before / now, K 128, N 2048: 8192 rows 24.1 / 17.6, 13971 40.7 / 27.7, 2000
    // 9.9 / 8.1; K 64, N 1024: 8192 14.3 / 12.0 (the fill of as many bytes: 11.0, 16.6, 5.1,
    // 7.2).
    const bool upper = l16 >= 8;
    const bool vec = (g.ldc & 3) == 0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int nt = 0; nt < NT; nt += 2) {
        const int nu = nt + 1 < NT ? nt + 1 : nt;
        const bool pair = nu > nt && nt0 + nu < n_tiles && vec &&
                          16 * (nt0 + nu + 1) <= g.n_store;
        if (pair) {
          float a[4], b[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = value(mt, nt, i), y = value(mt, nu, i);
            const float got = dpp_move<kDppRor8>(upper ? x : y);
            a[i] = upper ? got : x;
            b[i] = upper ? y : got;
          }
          const int n = 16 * (nt0 + nt) + 4 * gq + (upper ? 16 : 0);
          const int m = m0 + 16 * mt + (l16 & 7);
          float* o = g.C32 + (size_t)m * g.ldc + n;
          if (m < g.M) *reinterpret_cast<float4*>(o) = make_float4(a[0], a[1], a[2], a[3]);
          if (m + 8 < g.M)
            *reinterpret_cast<float4*>(o + (size_t)8 * g.ldc) = make_float4(b[0], b[1], b[2], b[3]);
          continue;
        }
        const int m = m0 + 16 * mt + l16;
        if (m >= g.M) continue;
#pragma unroll
        for (int u = nt; u <= nu; ++u) {
          if (nt0 + u >= n_tiles) continue;
          const int n = 16 * (nt0 + u) + 4 * gq;
          float* o = g.C32 + (size_t)m * g.ldc + n;
          if (vec && n + 4 <= g.n_store) {
            *reinterpret_cast<float4*>(o) = make_float4(value(mt, u, 0), value(mt, u, 1),
                                                        value(mt, u, 2), value(mt, u, 3));
            continue;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < g.n_store) o[i] = value(mt, u, i);
        }
      }
    }
    return;
  }
  if (DENSE == 1 || g.epilogue == T5D_EPI_GEGLU) {
    // tile columns 0..7 are wi_0, 8..15 the matching wi_1 columns: the lanes
    // with gq >= 2 hold the gates of the lanes with gq - 2.  32 output columns.
    // Two v_permlane32_swap hand every lane two (value, gate) pairs — the
    // lower half of the wavefront keeps its values 2, 3 and receives their
    // gates, the upper half keeps its gates 0, 1 and receives their values —
    // so all 64 lanes evaluate GELU on values that are used.
    const int F = g.N >> 1;
    const int row = lane / NT, piece = lane % NT;  // NT 16-byte pieces per row
    const bool lower = gq < 2;
    const int col0 = 4 * (gq & 1) + (lower ? 2 : 0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const auto a = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(value(mt, nt, 2)),
            __float_as_uint(value(mt, nt, 0)), false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(value(mt, nt, 3)),
            __float_as_uint(value(mt, nt, 1)), false, false);
        // [0]: the value (own in the lower half), [1]: its gate
        float h0, h1;
        if constexpr (DENSE == 1) {
          h0 = clamped_glu_bf16(__uint_as_float(a[0]), __uint_as_float(a[1]),
                           g.glu_limit, g.glu_alpha, g.glu_add);
          h1 = clamped_glu_bf16(__uint_as_float(b[0]), __uint_as_float(b[1]),
                           g.glu_limit, g.glu_alpha, g.glu_add);
        } else {
          h0 = round_bf16(gelu_sigmoid_form(round_bf16(__uint_as_float(a[0])))) *
               round_bf16(__uint_as_float(a[1]));
          h1 = round_bf16(gelu_sigmoid_form(round_bf16(__uint_as_float(b[0])))) *
               round_bf16(__uint_as_float(b[1]));
        }
        *reinterpret_cast<uint32_t*>(stage + l16 * 80 + (8 * nt + col0) * 2) =
            pack_bf16x2(h0, h1);
      }
      asm volatile("" ::: "memory");
      const uint4 q = *reinterpret_cast<const uint4*>(
          stage + min(row, 15) * 80 + piece * 16);
      asm volatile("" ::: "memory");
      const int m = m0 + 16 * mt + row;
      if (row < 16 && m < g.M && nt0 + piece < n_tiles)
        *reinterpret_cast<uint4*>(g.C + (size_t)m * F + 8 * (nt0 + piece)) = q;
    }
    return;
  }
  constexpr int PP = 2 * NT;    // 16-byte pieces per row of the slice
  constexpr int RPI = 64 / PP;  // rows per instruction (8, or 10 with 4 lanes idle)
  const int piece = lane % PP, prow = lane / PP;
  const int n = 16 * nt0 + 8 * piece;
  const bool n_ok = nt0 + (piece >> 1) < n_tiles;
  // The residual of AHEAD slices is under way while one is added (16384 x 768 x 768,
  // which waited for each slice: 31.9 -> 28.2 us with the bank conflicts gone too).
  constexpr int AHEAD = 4;
  const bool residual = NORM == 2 || g.epilogue == T5D_EPI_RESIDUAL;
  float next[8];
  if constexpr (NORM == 2) {
    const uint4 w = n_ok ? *reinterpret_cast<const uint4*>(g.next_scale + n)
                         : make_uint4(0, 0, 0, 0);
    unpack16(w, next);
  }
  uint4 res[AHEAD][2];
  const auto fetch = [&](int mt) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = m0 + 16 * mt + RPI * j + prow;
      res[mt % AHEAD][j] = make_uint4(0, 0, 0, 0);
      if (prow < RPI && RPI * j + prow < 16 && m < g.M && n_ok)
        res[mt % AHEAD][j] =
            *reinterpret_cast<const uint4*>(g.residual + (size_t)m * g.N + n);
    }
  };
  if (residual) {
#pragma unroll
    for (int mt = 0; mt < (AHEAD < MT ? AHEAD : MT); ++mt) fetch(mt);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<uint2*>(stage + l16 * kRowsStageStride<NT> + (16 * nt + 4 * gq) * 2) =
          pack4(value(mt, nt, 0), value(mt, nt, 1),
                value(mt, nt, 2), value(mt, nt, 3));
    asm volatile("" ::: "memory");
    uint4 back[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      back[j] = *reinterpret_cast<const uint4*>(
          stage + min(RPI * j + prow, 15) * kRowsStageStride<NT> + piece * 16);
    asm volatile("" ::: "memory");
    if (residual) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint4& q = back[j];
        const uint4 r = res[mt % AHEAD][j];
        q.x = pack_bf16x2(bf16lo_to_f32(q.x) + bf16lo_to_f32(r.x),
                          bf16hi_to_f32(q.x) + bf16hi_to_f32(r.x));
        q.y = pack_bf16x2(bf16lo_to_f32(q.y) + bf16lo_to_f32(r.y),
                          bf16hi_to_f32(q.y) + bf16hi_to_f32(r.y));
        q.z = pack_bf16x2(bf16lo_to_f32(q.z) + bf16lo_to_f32(r.z),
                          bf16hi_to_f32(q.z) + bf16hi_to_f32(r.z));
        q.w = pack_bf16x2(bf16lo_to_f32(q.w) + bf16lo_to_f32(r.w),
                          bf16hi_to_f32(q.w) + bf16hi_to_f32(r.w));
      }
      if (mt + AHEAD < MT) fetch(mt + AHEAD);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = RPI * j + prow;
      if (prow >= RPI || row >= 16) continue;
      const uint4 q = back[j];
      const int m = m0 + 16 * mt + row;
      if constexpr (NORM == 2) {
        float f[8];
        unpack16(q, f);
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
        ss = n_ok ? ss : 0.f;
        ss += dpp_move<kDppXor1>(ss);  // the tile's other 8 columns
        if ((piece & 1) == 0)
          shared[(wave * NT + (piece >> 1)) * (16 * MT) + 16 * mt + row] = ss;
        if (m < g.M && n_ok)
          *reinterpret_cast<uint4*>(g.scaled + (size_t)m * g.N + n) = make_uint4(
              pack_bf16x2(f[0] * next[0], f[1] * next[1]),
              pack_bf16x2(f[2] * next[2], f[3] * next[3]),
              pack_bf16x2(f[4] * next[4], f[5] * next[5]),
              pack_bf16x2(f[6] * next[6], f[7] * next[7]));
      }
      if (m >= g.M || !n_ok) continue;
      size_t o;
      if (g.layout == T5D_OUT_HEADS_KEY) {
        // [B, H, 2, Ep, 32]: the two 32-wide halves of the head dim as planes
        const int b = m / g.E, e = m - b * g.E;
        const int hh = n >> 6, c = (n >> 5) & 1, jj = n & 31;
        o = ((((size_t)b * g.H + hh) * 2 + c) * g.Ep + e) * 32 + jj;
      } else {
        o = (size_t)m * g.N + n;
      }
      *reinterpret_cast<uint4*>(g.C + o) = q;
    }
  }
}

// SWAP: weights are the MFMA A operand (C^T is formed).
template <typename WT, bool SWAP, int DENSE = 0>
__global__ void __launch_bounds__(256, 2)
rows_gemm_kernel(RowsGemmArgs g) {
  constexpr int TB = RowsWeightTile<WT>::kTileBytes;
  constexpr int MT = kRowsMT, NT = kRowsNT;
  // [buffer][tile][lane]: tiles 0..15 activations (rows 16 t ..), 16..23 weights
  __shared__ uint4 s_t[2][24][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, gq = lane >> 4;
  const int m_blocks = (g.M + kRowsBM - 1) / kRowsBM;
  const int m_blk = blockIdx.x % m_blocks, n_blk = blockIdx.x / m_blocks;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = m_blk * kRowsBM + wm * (16 * MT);
  const int nt0 = n_blk * (kRowsBN / 16) + wn * NT;  // first 16-column tile
  const int KT = g.K >> 5, n_tiles = g.N >> 4;

  // The 6 tiles this wavefront fetches: activation tiles wave + 4 i (i < 4),
  // weight tiles wave + 4 i (i < 2).  Out-of-range rows / tiles are clamped
  // (their products are discarded in the epilogue).
  // An activation tile is fetched with lane l reading piece l % 4 (8 k) of row
  // l / 4, so that four neighbouring lanes read 64 contiguous bytes: fetched in
  // operand order (lane = row + 16 * piece) every lane of a quarter wavefront
  // touches another row, 64 separate requests per instruction, and the L1's
  // tag lookups, not the matrix cores, set the pace.  The piece lands in LDS at
  // its operand slot, XOR-swizzled so that neither the parking writes nor the
  // operand reads collide on banks.
  const int ld_row = lane >> 2, ld_piece = lane & 3;
  const int park_slot = (ld_piece * 16 + ld_row) ^ (ld_piece * 2);
  const int read_slot = lane ^ (gq * 2);
  const bf16_t* arow[4];
  const char* wtile[2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    arow[i] = g.A +
              (size_t)min(m_blk * kRowsBM + 16 * (wave + 4 * i) + ld_row, g.M - 1) *
                  g.lda + 8 * ld_piece;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    wtile[i] = g.W + (size_t)min(n_blk * (kRowsBN / 16) + wave + 4 * i,
                                 n_tiles - 1) * KT * TB;

  f32x4_r acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = (f32x4_r){0.f, 0.f, 0.f, 0.f};

  // Staging registers of the 6 tiles in flight (named, not an array: they
  // must stay in registers across the loop).
  typedef typename RowsWeightTile<WT>::Raw RawW;
  uint4 sa0, sa1, sa2, sa3;
  RawW sw0, sw1;
#define T5D_ROWS_FETCH(kt_)                                                    \
  do {                                                                         \
    sa0 = *reinterpret_cast<const uint4*>(arow[0] + 32 * (kt_));               \
    sa1 = *reinterpret_cast<const uint4*>(arow[1] + 32 * (kt_));               \
    sa2 = *reinterpret_cast<const uint4*>(arow[2] + 32 * (kt_));               \
    sa3 = *reinterpret_cast<const uint4*>(arow[3] + 32 * (kt_));               \
    sw0 = RowsWeightTile<WT>::load(wtile[0] + (size_t)(kt_) * TB, lane);       \
    sw1 = RowsWeightTile<WT>::load(wtile[1] + (size_t)(kt_) * TB, lane);       \
  } while (0)
#define T5D_ROWS_PARK(buf_)                                                    \
  do {                                                                         \
    s_t[buf_][wave][park_slot] = sa0;                                          \
    s_t[buf_][wave + 4][park_slot] = sa1;                                      \
    s_t[buf_][wave + 8][park_slot] = sa2;                                      \
    s_t[buf_][wave + 12][park_slot] = sa3;                                     \
    s_t[buf_][16 + wave][lane] = RowsWeightTile<WT>::frag(sw0);                \
    s_t[buf_][20 + wave][lane] = RowsWeightTile<WT>::frag(sw1);                \
  } while (0)
  T5D_ROWS_FETCH(0);
  T5D_ROWS_PARK(0);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < KT) T5D_ROWS_FETCH(kt + 1);
    FragR wb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wb[nt].u = s_t[buf][16 + wn * NT + nt][lane];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      FragR xa;
      xa.u = s_t[buf][wm * MT + mt][read_slot];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if (SWAP)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wb[nt].v, xa.v, acc[mt][nt], 0, 0, 0);
        else
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              xa.v, wb[nt].v, acc[mt][nt], 0, 0, 0);
      }
    }
    if (kt + 1 < KT) T5D_ROWS_PARK(buf ^ 1);
    __syncthreads();
  }
#undef T5D_ROWS_FETCH
#undef T5D_ROWS_PARK

  if (SWAP) {
    // (the loop ends with a barrier: every wavefront is done with the tiles)
    static_assert(sizeof(s_t[0]) >= 4 * kRowsStageBytes<NT>, "stage too small");
    rows_epilogue_staged<DENSE, sizeof(WT) == 1>(
        g, acc, m0, nt0, n_tiles, lane,
        reinterpret_cast<char*>(&s_t[0][0][0]) + wave * kRowsStageBytes<NT>);
  } else {
    rows_epilogue_values(g, acc, m0, nt0, n_tiles, l16, gq);
  }
}

// ---- K >= 64: rows through LDS, weights into registers --------------------------
// A workgroup of 4 wavefronts owns BM = 16 MT rows x BN = 64 NT columns, a wavefront all
// rows of 16 NT columns.  So every weight is wanted by one wavefront only, and packed
// weights come in operand order: they go straight from memory into registers, two
// k-tiles of 32 ahead in three sets.  Rows are wanted by all four: they go straight into
// LDS (buffer_load ... lds, 16 bytes per lane), 64 of K at a time in a ring of three
// stages, whole 128-byte lines of 8 rows per instruction; one barrier per 64 of K.
// Operand reads from LDS run 16 rows ahead of the products, behind scheduling fences.
// Piece p of row r lies at slot p ^ (r / 2 % 8) of its 8: a 16-byte read serves lanes
// 0..3 and 12..15 of one quarter wavefront with 4..11 of its neighbour, which want
// the neighbouring piece, and these 16 then cover all banks.
//
// What bounds it, and why this split (measured, us; before: both operands through LDS,
// 32 of K per barrier, 256 x 256 by 8 wavefronts or 256 x 192 or 256 x 128):
//  - LDS: 128 x 64 per wavefront with both operands in LDS reads 24 KB and writes 8 KB
//    per 64 of K and wavefront, 2048 clocks of LDS beside 2048 of the matrix cores.
//    Weights in registers leave 1280.
//  - the order loads return in: a wavefront's loads come back as they were issued, so a
//    weight tile that is asked for behind rows that come from memory waits for them.
//    Rows are therefore requested in the middle of a step, behind the weights of the
//    next one (16384 x 768 x 768: 28.5 the other way round, 25.6 so).
//  - prologue and epilogue, which one workgroup per CU cannot cover: two or more share
//    one, each in its own phase.
//  16384 x 768 x 4096 gated 113.8 -> 92, 10300 x 768 x 4096 gated 77 -> 61, 10300 x 2048
//  x 768 46.7 -> 33, 5000 x 2816 x 1024 47 -> 34, 8192 x 1024 x 5632 gated 91 -> 81,
//  14000 x 1024 x 5632 gated 161 -> 132, 16384 x 4096 x 4096 412 -> 385 (1428 TFLOP/s;
//  matrix instructions alone, on random numbers, reach 2000 at the clock that is left
//  then), 2000 x 2048 x 768 16.9 -> 13, 1000 x 1024 x 5632 20.8 -> 14.3.  int8 weights,
//  widened in registers (before: 256 x 128 through staging registers): 8192 x 2048 x 2048
//  80 -> 65, 8192 x 5120 x 2048 175 -> 147, 1000 x 2816 x 1024 63 -> 22.
//
// Every wait is counted: the loop is straight-line code (rounds of three steps, as the
// ring and the register sets want; what is left over stands behind it), requests past
// the end ask for the last step again.  (global_load ... lds would do for rows, but the
// compiler takes it for a flat access, after which it waits for everything.)
// GROUPED: see GroupTiles (gemm_tiles.h); a tile of 256 rows is two workgroups.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_r;

typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_r;

// A weight tile's piece as a buffer load gives it, and as a matrix operand.
template <typename WT> struct RowsWeight;
template <> struct RowsWeight<bf16_t> {
  static constexpr int kTileBytes = 1024;
  u32x4_r raw;
#if defined(__HIP_DEVICE_COMPILE__)
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t from, int lane, int at) {
    raw = __builtin_amdgcn_raw_buffer_load_b128(from, 16 * lane, at, 0);
  }
#endif
  __device__ __forceinline__ bf16x8_r frag() const {
    return __builtin_bit_cast(bf16x8_r, raw);
  }
};
template <> struct RowsWeight<int8_t> {
  static constexpr int kTileBytes = 512;
  u32x2_r raw;
#if defined(__HIP_DEVICE_COMPILE__)
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t from, int lane, int at) {
    raw = __builtin_amdgcn_raw_buffer_load_b64(from, 8 * lane, at, 0);
  }
#endif
  __device__ __forceinline__ bf16x8_r frag() const {
    return __builtin_bit_cast(
        bf16x8_r, RowsWeightTile<int8_t>::frag(make_uint2(raw[0], raw[1])));
  }
};

// What a 32-bit offset of a buffer access reaches.
constexpr int64_t kRowsReach = 1LL << 31;

// The same products with operands fetched where they are used: for grouped layers whose
// rows or weights spread over more than a buffer access reaches.
template <int MT, int NT>
__device__ __forceinline__ void rows_multiply_far(const RowsGemmArgs& g,
                                                  f32x4_r (&acc)[MT][NT], int m0,
                                                  int nt0, int n_tiles, int lane) {
  const int l16 = lane & 15, gq = lane >> 4;
  const int KT = g.K >> 5;
  for (int kt = 0; kt < KT; ++kt) {
    FragR wb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      wb[nt].u = reinterpret_cast<const uint4*>(
          g.W + ((size_t)min(nt0 + nt, n_tiles - 1) * KT + kt) * 1024)[lane];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int row = group_row(g.grp, min(m0 + 16 * mt + l16, g.M - 1));
      FragR xa;
      xa.u = *reinterpret_cast<const uint4*>(g.A + (size_t)row * g.lda + 32 * kt +
                                             8 * gq);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[nt].v, xa.v,
                                                              acc[mt][nt], 0, 0, 0);
    }
  }
}

// FOLD: the sums of every step are added up apart from one another, as the kernels for
// few rows, in whose place this one then stands, add up those of their wavefronts:
// float32 results over K = 768, 1024, 2048 lie 8.3e-8, 9.4e-8, 1.31e-7 off the float64
// ones there, 1.57e-7, 1.84e-7, 2.71e-7 with one sum over all of K, 8.0e-8, 8.8e-8,
// 1.12e-7 so.
// NORM: the RMS norm between layers without a pass of its own.  2: rows with the residual
// added are stored as they are and times the norm's scale, with the sums of their squares,
// 64 columns each (the same additions whatever the tile); 1: A is such scaled rows, and
// results are divided by their root mean square, row by row.  The pass that this replaces
// read and wrote every row at 2 to 3 TB/s, 11.0 us for 10312 rows of 768, 9.9 for 4976 of
// 1024; the second store and the squares cost a layer 1 to 3 us.  Encoder of 12 layers of
// 768, 9372 rows, in passes of its own / inside 2541 / 2490 us, of 24 of 1024, 4896 rows,
// 4975 / 4890, both with everything else as it is here.
template <typename WT, bool SWAP, int MT, int NT, int DENSE, bool GROUPED, bool FOLD,
          int NORM>
__device__ __forceinline__ void rows_gemm_tile(
    const RowsGemmArgs& g, int m_blk, int n_blk, uint4 (&s_a0)[128 * MT],
    uint4 (&s_a1)[128 * MT], uint4 (&s_a2)[128 * MT], float* s_inv) {
#if defined(__HIP_DEVICE_COMPILE__)  // (buffer descriptors are no host type)
  constexpr int BM = 16 * MT, BN = 64 * NT;
  constexpr int TB = RowsWeight<WT>::kTileBytes;
  constexpr int AL = BM / 32;  // 1 KB pieces (8 rows) a wavefront loads per stage
  // Before every barrier: all but the newest rows and weights have landed (the stage
  // and the weight tile about to be multiplied), and my reads of LDS have returned.  A
  // barrier orders instructions that have been issued, not LDS reads that have
  // completed.
  constexpr int kWaitStage = 0x070 | (AL + NT);
  static_assert(AL + NT < 16, "vmcnt");
  constexpr int kWaitAll = 0x070;
  static_assert(sizeof(s_a0) >= 4 * kRowsStageBytes<NT>, "stage too small");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, gq = lane >> 4;
  const int KT = g.K >> 5, KS = (KT + 1) >> 1, n_tiles = g.N >> 4;
  const int m0 = m_blk * BM;
  const int nt0 = n_blk * (BN / 16) + wave * NT;
  constexpr int kSquares = NORM == 1 ? 16 : 1;
  float squares[kSquares], more[kSquares];
  const float* row_squares = nullptr;
  if constexpr (NORM == 1) {
    // requested in front of the operands, looked at behind their first requests; the
    // first barrier lies between here and the epilogue
    row_squares = g.squares_in + min(m0 + (int)(threadIdx.x & (BM - 1)), g.M - 1);
#pragma unroll
    for (int p = 0; p < kSquares; ++p)
      squares[p] = row_squares[(size_t)min(p, g.parts - 1) * g.M];
#pragma unroll
    for (int p = 0; p < kSquares; ++p) more[p] = 0.f;
    if (g.parts > kSquares) {
#pragma unroll
      for (int p = 0; p < kSquares; ++p)
        more[p] = row_squares[(size_t)min(kSquares + p, g.parts - 1) * g.M];
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  f32x4_r acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = (f32x4_r){0.f, 0.f, 0.f, 0.f};

  bool listed = false;
  if constexpr (GROUPED) {
    listed = g.grp.rows != nullptr;
    bool far = 2LL * BN * g.K >= kRowsReach || 2LL * (BM + 1) * g.lda >= kRowsReach;
    if (listed) {
      const int reach = (int)((kRowsReach - 1) / (2LL * g.lda)) - 1;
#pragma unroll
      for (int r = 0; r < BM; r += 64)
        far |= g.grp.rows[min(m0 + r + lane, g.M - 1)] > reach;
    }
    if (__builtin_amdgcn_ballot_w64(far) != 0) {
      rows_multiply_far(g, acc, m0, nt0, n_tiles, lane);
      rows_epilogue_staged<DENSE, false>(
          g, acc, m0, nt0, n_tiles, lane,
          reinterpret_cast<char*>(&s_a0[0]) + wave * kRowsStageBytes<NT>);
      return;
    }
  }
  // this wavefront's pieces of every stage: 8-row groups wave + 4 i (rows past the edge
  // clamped: their products are discarded in the epilogue)
  const __amdgpu_buffer_rsrc_t a_rows = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(listed ? g.A : g.A + (size_t)m0 * g.lda), 0, 0x7fffffff, 0x00020000);
  const int ld_row = wave * 8 + (lane >> 3);
  const int ld_piece = (lane & 7) ^ ((ld_row >> 1) & 7);  // (32 rows on: the same)
  int a_off[AL];
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    const int row = min(m0 + ld_row + 32 * i, g.M - 1);
    a_off[i] = (listed ? group_row(g.grp, row) : row - m0) * (g.lda * 2) + 16 * ld_piece;
  }
  // K of 32 modulo 64: the last step has no second half, whose pieces are the first's
  const int a_back = (KT & 1) && ld_piece >= 4 ? 64 : 0;
  const __amdgpu_buffer_rsrc_t w_rows = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(g.W + (size_t)n_blk * (BN / 16) * KT * TB), 0, 0x7fffffff, 0x00020000);
  int w_off[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    w_off[nt] = min(wave * NT + nt, n_tiles - 1 - n_blk * (BN / 16)) * KT * TB;
  RowsWeight<WT> w0[NT], w1[NT], w2[NT];

#define T5D_ROWS_ISSUE_A(s_, S_)                                               \
  do {                                                                         \
    const int step = min((s_), KS - 1);                                        \
    const int back = step == KS - 1 ? a_back : 0;                              \
    _Pragma("unroll") for (int i = 0; i < AL; ++i)                             \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(                                \
          a_rows, (lds_ptr_t)&S_[(wave + 4 * i) * 64], 16, a_off[i] - back,    \
          128 * step, 0, 0);                                                   \
  } while (0)
#define T5D_ROWS_ISSUE_W(kt_, W_)                                              \
  _Pragma("unroll") for (int nt = 0; nt < NT; ++nt)                            \
    W_[nt].load(w_rows, lane, w_off[nt] + min((kt_), KT - 1) * TB)
#define T5D_ROWS_READ(S_, half_, p_, X_)                                       \
  _Pragma("unroll") for (int j = 0; j < 2; ++j)                                \
    X_[j].u = S_[(2 * (p_) + j) * 128 + l16 * 8 +                              \
                 ((4 * (half_) + gq) ^ ((l16 >> 1) & 7))]
#define T5D_ROWS_PRODUCTS(p_, X_, W_)                                          \
  _Pragma("unroll") for (int j = 0; j < 2; ++j)                                \
    _Pragma("unroll") for (int nt = 0; nt < NT; ++nt)                          \
      acc[2 * (p_) + j][nt] =                                                  \
          SWAP ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(                      \
                     W_[nt], X_[j].v, acc[2 * (p_) + j][nt], 0, 0, 0)          \
               : __builtin_amdgcn_mfma_f32_16x16x32_bf16(                      \
                     X_[j].v, W_[nt], acc[2 * (p_) + j][nt], 0, 0, 0)
#define T5D_FENCE __builtin_amdgcn_sched_barrier(0)
  // Half a step: operands in x at its start, those of what follows in x at its end.
#define T5D_ROWS_HALF(S_, half_, W_)                                           \
  _Pragma("unroll") for (int nt = 0; nt < NT; ++nt) wf[nt] = W_[nt].frag();    \
  _Pragma("unroll") for (int p = 0; p < MT / 2; p += 2) {                      \
    T5D_ROWS_READ(S_, half_, p + 1, y);                                        \
    T5D_FENCE;                                                                 \
    T5D_ROWS_PRODUCTS(p, x, wf);                                               \
    T5D_FENCE;                                                                 \
    if (p + 2 < MT / 2) T5D_ROWS_READ(S_, half_, p + 2, x);                    \
    else if ((half_) == 0) T5D_ROWS_READ(S_, 1, 0, x);                         \
    T5D_FENCE;                                                                 \
    T5D_ROWS_PRODUCTS(p + 1, y, wf);                                           \
    T5D_FENCE;                                                                 \
  }
  // Step s_ on stage CUR_ with weights WA_, WB_; WC_, then WA_ take the next step's.
#define T5D_ROWS_STEP(s_, CUR_, NEXT2_, WA_, WB_, WC_, second_half_)           \
  do {                                                                         \
    FragR x[2], y[2];                                                          \
    bf16x8_r wf[NT];                                                           \
    __builtin_amdgcn_s_waitcnt(kWaitStage);                                    \
    __builtin_amdgcn_s_barrier();                                              \
    T5D_ROWS_READ(CUR_, 0, 0, x);                                              \
    T5D_FENCE;                                                                 \
    T5D_ROWS_ISSUE_W(2 * (s_) + 2, WC_);                                       \
    T5D_FENCE;                                                                 \
    T5D_ROWS_HALF(CUR_, 0, WA_)                                                \
    T5D_ROWS_ISSUE_W(2 * (s_) + 3, WA_);                                       \
    T5D_ROWS_ISSUE_A((s_) + 2, NEXT2_);                                        \
    T5D_FENCE;                                                                 \
    if (second_half_) {                                                        \
      T5D_ROWS_HALF(CUR_, 1, WB_)                                              \
    }                                                                          \
  } while (0)
  T5D_ROWS_ISSUE_A(0, s_a0);
  T5D_ROWS_ISSUE_W(0, w0);
  T5D_ROWS_ISSUE_W(1, w1);
  T5D_ROWS_ISSUE_A(1, s_a1);
  T5D_FENCE;
  if constexpr (NORM == 1) {
    float sum = squares[0];
#pragma unroll
    for (int p = 1; p < kSquares; ++p) sum += p < g.parts ? squares[p] : 0.f;
#pragma unroll
    for (int p = 0; p < kSquares; ++p) sum += kSquares + p < g.parts ? more[p] : 0.f;
    for (int p = 2 * kSquares; p < g.parts; ++p) sum += row_squares[(size_t)p * g.M];
    if (threadIdx.x < BM)
      s_inv[threadIdx.x] = 1.0f / sqrtf(sum / g.norm_d + g.eps);
    T5D_FENCE;
  }
  f32x4_r sums[FOLD ? MT : 1][FOLD ? NT : 1];
  if constexpr (FOLD) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) sums[mt][nt] = acc[mt][nt];
  }
  const auto fold = [&] {
    if constexpr (FOLD) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          sums[mt][nt] += acc[mt][nt];
          acc[mt][nt] = (f32x4_r){0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  int s = 0;
  for (; s + 3 <= KT >> 1; s += 3) {
    T5D_ROWS_STEP(s, s_a0, s_a2, w0, w1, w2, true);
    fold();
    T5D_ROWS_STEP(s + 1, s_a1, s_a0, w2, w0, w1, true);
    fold();
    T5D_ROWS_STEP(s + 2, s_a2, s_a1, w1, w2, w0, true);
    fold();
  }
  // the last 0 to 3 steps
  if (s < KS) {
    T5D_ROWS_STEP(s, s_a0, s_a2, w0, w1, w2, 2 * s + 1 < KT);
    if (s + 1 < KS) {
      T5D_ROWS_STEP(s + 1, s_a1, s_a0, w2, w0, w1, 2 * s + 3 < KT);
      if (s + 2 < KS) T5D_ROWS_STEP(s + 2, s_a2, s_a1, w1, w2, w0, 2 * s + 5 < KT);
    }
  }
#undef T5D_ROWS_ISSUE_A
#undef T5D_ROWS_ISSUE_W
#undef T5D_ROWS_READ
#undef T5D_ROWS_PRODUCTS
#undef T5D_FENCE
#undef T5D_ROWS_HALF
#undef T5D_ROWS_STEP
  if constexpr (FOLD) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] += sums[mt][nt];
  }
  if (SWAP) {
    // the requests past the end have landed, every wavefront is done with the ring
    __builtin_amdgcn_s_waitcnt(kWaitAll);
    __syncthreads();
    float* shared = NORM == 1 ? s_inv : reinterpret_cast<float*>(&s_a1[0]);
    static_assert(sizeof(s_a1) >= BN / 16 * BM * sizeof(float), "squares too many");
    rows_epilogue_staged<DENSE, sizeof(WT) == 1, MT, NT, NORM>(
        g, acc, m0, nt0, n_tiles, lane,
        reinterpret_cast<char*>(&s_a0[0]) + wave * kRowsStageBytes<NT>, shared, wave);
    if constexpr (NORM == 2) {
      __syncthreads();
      for (int i = threadIdx.x; i < NT * BM; i += 256) {
        const int group = i / BM, row = i % BM;
        const float* t = shared + 4 * group * BM + row;
        const int m = m0 + row, at = n_blk * NT + group;
        if (m < g.M && 64 * at < g.N)
          g.squares_out[(size_t)at * g.M + m] =
              (t[0] + t[BM]) + (t[2 * BM] + t[3 * BM]);
      }
    }
  } else {
    __builtin_amdgcn_s_waitcnt(kWaitAll);
    rows_epilogue_values(g, acc, m0, nt0, n_tiles, l16, gq,
                         NORM == 1 ? s_inv : nullptr);
  }
#endif
}

// An XCD takes a run of consecutive tiles, column by column over 8 blocks of rows at a
// time: what its CUs hold at once is few rows and few weights.
__device__ __forceinline__ void rows_tile_of(int m_blocks, int n_blocks, int& m_blk,
                                             int& n_blk) {
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int total = m_blocks * n_blocks;
  const int t = xcd * (total >> 3) + min(xcd, total & 7) + slot;
  constexpr int GM = 8;
  const int group = t / (GM * n_blocks), in = t - group * (GM * n_blocks);
  const int rows = min(GM, m_blocks - group * GM);
  m_blk = group * GM + in % rows;
  n_blk = in / rows;
}

template <typename WT, bool SWAP, int MT, int NT, int OCC, int DENSE = 0,
          bool GROUPED = false, bool FOLD = false, int NORM = 0>
__global__ void __launch_bounds__(256, OCC)
rows_gemm_direct_kernel(RowsGemmArgs g) {
  constexpr int BM = 16 * MT, BN = 64 * NT;
  __shared__ uint4 s_a0[BM * 8];
  __shared__ uint4 s_a1[BM * 8];
  __shared__ uint4 s_a2[BM * 8];
  __shared__ __align__(16) float s_inv[NORM == 1 ? BM : 4];
  T5D_GATED(g.gate);
  const int n_blocks = ((g.N >> 4) + BN / 16 - 1) / (BN / 16);
  int m_blk, n_blk;
  if constexpr (GROUPED) {
    // 4 consecutive tiles of rows, most of them of one group, on one XCD, all
    // columns of half a tile in a row: rows and kernels come from that XCD's L2.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int t = slot / n_blocks;
    const int tile = ((t >> 3) * 8 + xcd) * 4 + ((t & 7) >> 1);
    m_blk = t & 1;
    n_blk = slot % n_blocks;
    if (tile >= g.n_tiles ||
        !enter_group(g.grp, tile, g.A, g.lda, g.W, g.C, DENSE == 1 ? g.N >> 1 : g.N,
                     g.M) ||
        m_blk * BM >= g.M)
      return;
  } else {
    rows_tile_of((g.M + BM - 1) / BM, n_blocks, m_blk, n_blk);
  }
  rows_gemm_tile<WT, SWAP, MT, NT, DENSE, GROUPED, FOLD, NORM>(g, m_blk, n_blk, s_a0,
                                                               s_a1, s_a2, s_inv);
}

// Two layers over the same rows in one launch, the second into the value layout: an
// encoder's q | k and v, which are too narrow to fill the rounds of workgroups each on its
// own (see rows_pair).
template <typename WT, int MT, int NT, int OCC, int NORM>
__global__ void __launch_bounds__(256, OCC)
rows_gemm_pair_kernel(RowsGemmArgs g) {
  constexpr int BM = 16 * MT, BN = 64 * NT;
  __shared__ uint4 s_a0[BM * 8];
  __shared__ uint4 s_a1[BM * 8];
  __shared__ uint4 s_a2[BM * 8];
  __shared__ __align__(16) float s_inv[NORM == 1 ? BM : 4];
  const int n1 = (g.N + BN - 1) / BN, n2 = (g.N2 + BN - 1) / BN;
  int m_blk, n_blk;
  rows_tile_of((g.M + BM - 1) / BM, n1 + n2, m_blk, n_blk);
  if (n_blk < n1) {
    g.layout = T5D_OUT_ROWS;
    rows_gemm_tile<WT, true, MT, NT, 0, false, false, NORM>(g, m_blk, n_blk, s_a0, s_a1,
                                                            s_a2, s_inv);
  } else {
    g.W = g.W2;
    g.scales = g.scales2;
    g.C = g.C2;
    g.N = g.N2;
    rows_gemm_tile<WT, false, MT, NT, 0, false, false, NORM>(g, m_blk, n_blk - n1, s_a0,
                                                             s_a1, s_a2, s_inv);
  }
}

}  // namespace t5d

using namespace t5d;

// The workgroup tile of rows_gemm_direct_kernel: 128 rows x 256, 192 or 128 columns, or
// 64 x 128; 2, 2, 3 and 4 of them share a CU.  What a step of 64 of K lasts (us) with
// 1, 2, ... of a kind on each CU, fitted to M = 1000 .. 32768, K = 768 .. 4096, N = 768
// .. 8192: a lone workgroup waits for its operands, several overlap, and beyond that
// time goes by their area.  The tile whose rounds over the 256 CUs add up to least is
// taken.  Measured, us, 256 / 192 / 128 columns / 64 rows (* taken):
//   10300 x 768 x 768 residual  18.3 / 21.6 / 17.9* / 18.2
//   5000 x 2816 x 1024          38.5 / 33.6* / 37.3 / 38.8
//   2000 x 2048 x 768           28.4 / 24.1 / 18.0 / 12.9*
//   4096 x 1024 x 1024          15.8 / 13.8 / 10.6* / 10.9
//   14000 x 1024 x 1024         28.0* / 33.0 / 30.2 / 34.1
//   16384 x 768 x 4096 gated    92* / 96 / 95 / 117
//   16384 x 768 x 1536          34 / 37* / 36 / 45
struct RowsTile {
  int code, rows, cols, per_cu;
  double step[4];
};
static const RowsTile kRowsTiles[] = {
    {2, 128, 256, 2, {0.77, 1.30}},
    {3, 128, 192, 2, {0.56, 1.03}},
    {1, 128, 128, 3, {0.42, 0.755, 1.15}},
    {1, 64, 128, 4, {0.28, 0.45, 0.80, 1.00}},
};

// N2: columns of a second layer in the same launch.  Where all of the layer is one round of
// lone workgroups of 256 columns, they read the rows half as often as the two of 128 columns
// per CU, which counts for more than their overlap once the rows are more than the L2s keep.
// us, 128 / 256 columns, rows x K x N (plain; with residual and norm):
//   6360 x 1536 x 1024 (20 MB)  24.2 / 24.6; 28.5 / 29.0    7256 (22 MB)  26.8 / 24.9; 32.2 / 30.1
//   9688 x 1024 x 768  (20 MB)  20.1 / 19.7; 25.0 / 24.2   10840 (22 MB)  21.3 / 20.0; 27.6 / 25.0
//   3160 x 2816 x 2048 (18 MB)  38.3 / 37.9; 42.5 / 42.4    4056 (23 MB)  44.0 / 41.6; 49.6 / 47.2
//   8152 x 2816 x 1024 (46 MB)  48.3 / 42.8; 52.5 / 48.0
//   10840 x 2048 x 768 (44 MB)  40.7 / 33.5; 46.8 / 39.8
//   3160 x 1024 x 2048 (6 MB)   17.5 / 18.4; 20.6 / 23.1
static double rows_tile_cost(const RowsTile& t, int64_t M, int K, int N, int N2 = 0) {
  const int64_t wgs = ((M + t.rows - 1) / t.rows) *
                      ((N + t.cols - 1) / t.cols + (N2 + t.cols - 1) / t.cols);
  if (t.cols == 256 && wgs <= 256 && 2 * M * K >= 22000000) return 0.70;
  const int64_t slots = 256 * t.per_cu, left = wgs % slots;
  return (double)(wgs / slots) * t.step[t.per_cu - 1] +
         (left ? t.step[(left + 255) / 256 - 1] : 0.0);
}

// Whether the kernel takes the shape (offsets inside a workgroup's rows and weights are
// 32 bits wide), else rows_gemm_kernel does.
static bool rows_direct(int K, int64_t lda) {
  return K >= 64 && 2LL * 256 * K < kRowsReach &&
         2LL * 128 * lda + 2LL * K < kRowsReach;
}

// code 0: any.
static const RowsTile& rows_tile(int64_t M, int K, int N, int code, int N2 = 0) {
  const RowsTile* best = nullptr;
  double least = 0.0;
  for (const RowsTile& t : kRowsTiles) {
    if (code && t.code != code) continue;
    const double c = rows_tile_cost(t, M, K, N, N2);
    if (best == nullptr || c < least) {
      best = &t;
      least = c;
    }
  }
  return *best;
}

extern "C" int t5d_gemm_rows_tile(int w_dtype, int64_t M, int K, int N) {
  if (w_dtype != T5D_BF16 || M <= 0 || N <= 0 || K <= 0 || !rows_direct(K, K)) return 1;
  return rows_tile(M, K, N, 0).code;
}

template <bool SWAP, int DENSE, int NORM = 0>
static void launch_rows_direct(hipStream_t s, const RowsGemmArgs& g, int w_dtype,
                               int code) {
  // (int8 weights, which are widened in registers on their way to the matrix cores, have
  // the tiles of 128 columns only)
  const RowsTile& t = rows_tile(g.M, g.K, g.N, w_dtype == T5D_I8 ? 1 : code);
  const dim3 grid((unsigned)((g.M + t.rows - 1) / t.rows) *
                  ((g.N + t.cols - 1) / t.cols));
#define T5D_ROWS_LAUNCH(WT_, MT_, NT_, OCC_)                                     \
  hipLaunchKernelGGL((rows_gemm_direct_kernel<WT_, SWAP, MT_, NT_, OCC_, DENSE,  \
                                              false, false, NORM>),              \
                     grid, dim3(256), 0, s, g)
  if constexpr (DENSE == 0 && NORM == 0) {
    if (w_dtype == T5D_I8) {
      if (t.rows == 64) T5D_ROWS_LAUNCH(int8_t, 4, 2, 4);
      else T5D_ROWS_LAUNCH(int8_t, 8, 2, 3);
      return;
    }
  }
  if (t.rows == 64) T5D_ROWS_LAUNCH(bf16_t, 4, 2, 4);
  else if (t.cols == 128) T5D_ROWS_LAUNCH(bf16_t, 8, 2, 3);
  else if (t.cols == 192) T5D_ROWS_LAUNCH(bf16_t, 8, 3, 2);
  else T5D_ROWS_LAUNCH(bf16_t, 8, 4, 2);
#undef T5D_ROWS_LAUNCH
}

// The workgroup tile of two layers in one launch; null: two launches.  Over up to 768
// inputs that is 128 columns: with 64 to 768 inputs and 128 to 32768 rows it is within 4 %
// of the fastest, but that 256 lead by 5 % over 16384 rows of 512 + 512 columns and more.
// us, 128 / 192 / 256 columns; two launches (rows x inputs, thrice as many columns):
//    2048 x 384   8.8 / 11.0 / 13.2; 10.1     10304 x 640  33.8 / 36.1 / 34.5; 37.6
//   10304 x 384  16.8 / 17.5 / 19.7; 20.3     10304 x 768  41.2 / 43.1 / 43.0; 44.0
//    4096 x 512  13.2 / 16.4 / 15.8; 14.1     16384 x 768  61.1 / 59.9 / 59.9; 64.1
//   16384 x 512  33.3 / 37.1 / 31.6; 35.9     24576 x 768  88.0 / 89.3 / 89.0; 92.4
// One launch gains
// where the two leave part of a round empty; beyond five rounds, and where the cost model
// says that the two fit their rounds better, there are two.  us, two launches / one (rows x
// inputs x columns + columns):
//    1024 x  512 x  768 + 384   20.9 / 12.3      4096 x  768 x 1536 + 768   25.0 / 21.5
//   10304 x  768 x 1536 + 768   42.3 / 41.0     12288 x  768 x 1536 + 768   50.7 / 46.2
//   24576 x  768 x 1536 + 768   90.2 / 84.7     32768 x  768 x 1536 + 768    110 / 113*
//    4992 x 1024 x 2048 + 1024  41.9 / 34.7     10304 x 1024 x 2048 + 1024  70.7 / 62.7
//   12288 x 1024 x 2048 + 1024  70.7 / 73.6*    16384 x 1024 x 2048 + 1024  91.9 / 88.6
//    6144 x 2048 x 4096 + 2048   128 / 131*     10304 x 2048 x 4096 + 2048   233 / 210
// (* two are launched).
static const RowsTile* rows_pair(const RowsGemmArgs& g, int w_dtype, int code) {
  const bool narrow = g.K <= 768;
  const RowsTile& t =
      rows_tile(g.M, g.K, g.N, w_dtype == T5D_I8 || (code == 0 && narrow) ? 1 : code,
                g.N2);
  if (code != 0) return &t;
  const int64_t wgs = (int64_t)((g.M + t.rows - 1) / t.rows) *
                      ((g.N + t.cols - 1) / t.cols + (g.N2 + t.cols - 1) / t.cols);
  if (wgs > 5 * 256 * t.per_cu) return nullptr;
  if (!narrow && wgs > 2 * 256 * t.per_cu) {
    const int any = w_dtype == T5D_I8 ? 1 : 0;
    const double apart = rows_tile_cost(rows_tile(g.M, g.K, g.N, any), g.M, g.K, g.N) +
                         rows_tile_cost(rows_tile(g.M, g.K, g.N2, any), g.M, g.K, g.N2);
    if (rows_tile_cost(t, g.M, g.K, g.N, g.N2) > 1.03 * apart) return nullptr;
  }
  return &t;
}

template <int NORM>
static void launch_rows_pair(hipStream_t s, const RowsGemmArgs& g, int w_dtype, int code) {
  const RowsTile* tile = rows_pair(g, w_dtype, code);
  if (tile == nullptr) {
    RowsGemmArgs one = g;
    one.layout = T5D_OUT_ROWS;
    launch_rows_direct<true, 0, NORM>(s, one, w_dtype, 0);
    one.layout = T5D_OUT_HEADS_VALUE;
    one.W = g.W2; one.scales = g.scales2; one.C = g.C2; one.N = g.N2;
    launch_rows_direct<false, 0, NORM>(s, one, w_dtype, 0);
    return;
  }
  const RowsTile& t = *tile;
  const dim3 grid((unsigned)((g.M + t.rows - 1) / t.rows) *
                  ((g.N + t.cols - 1) / t.cols + (g.N2 + t.cols - 1) / t.cols));
#define T5D_ROWS_LAUNCH(WT_, MT_, NT_, OCC_)                                     \
  hipLaunchKernelGGL((rows_gemm_pair_kernel<WT_, MT_, NT_, OCC_, NORM>), grid,   \
                     dim3(256), 0, s, g)
  if constexpr (NORM == 0) {
    if (w_dtype == T5D_I8) {
      if (t.rows == 64) T5D_ROWS_LAUNCH(int8_t, 4, 2, 4);
      else T5D_ROWS_LAUNCH(int8_t, 8, 2, 3);
      return;
    }
  }
  if (t.rows == 64) T5D_ROWS_LAUNCH(bf16_t, 4, 2, 4);
  else if (t.cols == 128) T5D_ROWS_LAUNCH(bf16_t, 8, 2, 3);
  else if (t.cols == 192) T5D_ROWS_LAUNCH(bf16_t, 8, 3, 2);
  else T5D_ROWS_LAUNCH(bf16_t, 8, 4, 2);
#undef T5D_ROWS_LAUNCH
}

// Picks the kernel and its workgroup tile (tile 0) and launches checked arguments.
static int launch_rows(hipStream_t s, int w_dtype, const RowsGemmArgs& g,
                       int tile) {
  const int m_blocks = (g.M + kRowsBM - 1) / kRowsBM;
  const int n_blocks = (g.N + kRowsBN - 1) / kRowsBN;
  const dim3 grid((unsigned)m_blocks * n_blocks), block(256);
  const bool swap = g.layout != T5D_OUT_HEADS_VALUE;
  const int dense = g.epilogue == T5D_EPI_CLAMPED_GLU ? 1 : g.C32 != nullptr ? 2 : 0;
  if (g.N2 > 0) {  // (rows_direct is the caller's)
    if (g.squares_in != nullptr) launch_rows_pair<1>(s, g, w_dtype, tile);
    else launch_rows_pair<0>(s, g, w_dtype, tile);
  } else if (g.squares_in != nullptr) {
    if (swap) launch_rows_direct<true, 0, 1>(s, g, w_dtype, tile);
    else launch_rows_direct<false, 0, 1>(s, g, w_dtype, tile);
  } else if (g.squares_out != nullptr) {
    launch_rows_direct<true, 0, 2>(s, g, w_dtype, tile);
  } else if (rows_direct(g.K, g.lda)) {
    if (dense == 1) launch_rows_direct<true, 1>(s, g, w_dtype, tile);
    else if (dense == 2) launch_rows_direct<true, 2>(s, g, w_dtype, tile);
    else if (swap) launch_rows_direct<true, 0>(s, g, w_dtype, tile);
    else launch_rows_direct<false, 0>(s, g, w_dtype, tile);
  } else if (dense == 1) {
    hipLaunchKernelGGL((rows_gemm_kernel<bf16_t, true, 1>), grid, block, 0, s, g);
  } else if (dense == 2) {
    hipLaunchKernelGGL((rows_gemm_kernel<bf16_t, true, 2>), grid, block, 0, s, g);
  } else if (w_dtype == T5D_BF16) {
    if (swap)
      hipLaunchKernelGGL((rows_gemm_kernel<bf16_t, true>), grid, block, 0, s, g);
    else
      hipLaunchKernelGGL((rows_gemm_kernel<bf16_t, false>), grid, block, 0, s, g);
  } else {
    if (swap)
      hipLaunchKernelGGL((rows_gemm_kernel<int8_t, true>), grid, block, 0, s, g);
    else
      hipLaunchKernelGGL((rows_gemm_kernel<int8_t, false>), grid, block, 0, s, g);
  }
  T5D_CHECK_LAUNCH("t5d_gemm_rows");
  return T5D_OK;
}

extern "C" int t5d_gemm_rows(void* stream, int w_dtype, const void* A,
                             const void* W, const float* scales,
                             const void* residual, void* C, int64_t M, int K,
                             int N, int epilogue, int out_layout, int E,
                             int Ep) {
  return t5d_gemm_rows_tiled(stream, w_dtype, A, W, scales, residual, C, M, K,
                             N, epilogue, out_layout, E, Ep, 0);
}

static int gemm_rows(void* stream, int w_dtype, const void* A, const void* W,
                     const float* scales, const void* residual, void* C, int64_t M,
                     int K, int N, int epilogue, int out_layout, int E, int Ep,
                     const int32_t* at, int tile, const t5d_rows_norm* norm = nullptr,
                     const t5d_rows_second* second = nullptr) {
  T5D_REQUIRE(A && W && C, T5D_EINVAL, "t5d_gemm_rows: null pointer");
  T5D_REQUIRE(tile >= 0 && tile <= 3, T5D_EINVAL,
              "t5d_gemm_rows_tiled: tile %d (0 chosen here, columns: 1: 128, "
              "2: 256, 3: 192)", tile);
  T5D_REQUIRE(w_dtype == T5D_BF16 || w_dtype == T5D_I8, T5D_EINVAL,
              "t5d_gemm_rows: w_dtype %d (packed bfloat16 or int8)", w_dtype);
  T5D_REQUIRE(w_dtype != T5D_I8 || scales, T5D_EINVAL,
              "t5d_gemm_rows: int8 weights need scales");
  T5D_REQUIRE(M > 0 && M < (1 << 30) && K > 0 && K % 32 == 0 && N > 0 &&
                  N % 16 == 0,
              T5D_EINVAL, "t5d_gemm_rows: M=%lld K=%d N=%d (K %% 32, N %% 16)",
              (long long)M, K, N);
  T5D_REQUIRE(epilogue >= T5D_EPI_NONE && epilogue <= T5D_EPI_GEGLU, T5D_EINVAL,
              "t5d_gemm_rows: epilogue %d", epilogue);
  T5D_REQUIRE(epilogue != T5D_EPI_RESIDUAL || residual, T5D_EINVAL,
              "t5d_gemm_rows: residual epilogue without residual");
  T5D_REQUIRE(out_layout >= T5D_OUT_ROWS && out_layout <= T5D_OUT_HEADS_VALUE,
              T5D_EINVAL, "t5d_gemm_rows: out_layout %d", out_layout);
  T5D_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 &&
                  ((uintptr_t)C % 8) == 0 && ((uintptr_t)residual % 8) == 0,
              T5D_EINVAL, "t5d_gemm_rows: operand alignment");
  int H = 0;
  if (out_layout != T5D_OUT_ROWS) {
    T5D_REQUIRE(epilogue == T5D_EPI_NONE && (second ? second->N : N) % 64 == 0 &&
                    E > 0 && Ep >= E &&
                    (at ? M % 4 == 0 : M % E == 0 && E % 4 == 0) && Ep % 32 == 0,
                T5D_EINVAL,
                "t5d_gemm_rows: heads layout needs epilogue none, N %% 64 == 0,"
                " M %% E == 0, E %% 4 == 0, Ep %% 32 == 0 (N=%d E=%d Ep=%d)", N,
                E, Ep);
    H = (second ? second->N : N) / 64;
  }
  RowsGemmArgs g = {};
  g.A = (const bf16_t*)A; g.W = (const char*)W;
  g.scales = w_dtype == T5D_I8 ? scales : nullptr;
  g.residual = (const bf16_t*)residual; g.C = (bf16_t*)C;
  g.M = (int)M; g.K = K; g.N = N;
  g.epilogue = epilogue; g.layout = out_layout;
  g.E = E; g.Ep = Ep; g.H = H; g.at = at;
  g.lda = K; g.C32 = nullptr; g.ldc = g.n_store = N;
  g.glu_limit = g.glu_alpha = g.glu_add = 0.f;
  g.gate = nullptr; g.grp = GroupTiles(); g.n_tiles = 0;
  if (norm != nullptr) {
    T5D_REQUIRE(rows_direct(K, K), T5D_ELIMIT, "t5d_gemm_rows_normed: K=%d", K);
    T5D_REQUIRE(w_dtype == T5D_BF16, T5D_EINVAL, "t5d_gemm_rows_normed: w_dtype %d",
                w_dtype);
    T5D_REQUIRE(norm->squares && (norm->scale == nullptr) == (norm->scaled == nullptr) &&
                    ((uintptr_t)norm->scale % 16) == 0 &&
                    ((uintptr_t)norm->scaled % 16) == 0,
                T5D_EINVAL, "t5d_gemm_rows_normed: norm buffers");
    T5D_REQUIRE(norm->scale ? epilogue == T5D_EPI_RESIDUAL
                            : epilogue != T5D_EPI_RESIDUAL && norm->eps > 0.f,
                T5D_EINVAL, "t5d_gemm_rows_normed: epilogue %d, eps %f", epilogue,
                (double)norm->eps);
    if (norm->scale) {
      T5D_REQUIRE(((uintptr_t)C % 16) == 0 && ((uintptr_t)residual % 16) == 0, T5D_EINVAL,
                  "t5d_gemm_rows_normed: operand alignment");
      g.next_scale = (const bf16_t*)norm->scale; g.scaled = (bf16_t*)norm->scaled;
      g.squares_out = norm->squares;
    } else {
      g.squares_in = norm->squares; g.parts = (K + 63) / 64;
      g.norm_d = (float)K; g.eps = norm->eps;
    }
  }
  if (second != nullptr) {
    T5D_REQUIRE(rows_direct(K, K), T5D_ELIMIT, "t5d_gemm_rows_pair: K=%d", K);
    T5D_REQUIRE(second->W && second->C && second->N > 0 &&
                    (w_dtype != T5D_I8 || second->scales) &&
                    ((uintptr_t)second->W % 16) == 0 && ((uintptr_t)second->C % 8) == 0 &&
                    ((uintptr_t)C % 16) == 0 && (!norm || !norm->scale),
                T5D_EINVAL, "t5d_gemm_rows_pair: second layer, N=%d", second->N);
    g.W2 = (const char*)second->W; g.C2 = (bf16_t*)second->C; g.N2 = second->N;
    g.scales2 = w_dtype == T5D_I8 ? second->scales : nullptr;
  }
  return launch_rows(as_stream(stream), w_dtype, g, tile);
}

extern "C" int t5d_gemm_rows_pair(void* stream, int w_dtype, const void* A, const void* W,
                                  const float* scales, void* C, int64_t M, int K, int N,
                                  int E, int Ep, const int32_t* at, int tile,
                                  const t5d_rows_second* second,
                                  const t5d_rows_norm* norm) {
  T5D_REQUIRE(second, T5D_EINVAL, "t5d_gemm_rows_pair: null pointer");
  return gemm_rows(stream, w_dtype, A, W, scales, nullptr, C, M, K, N, T5D_EPI_NONE,
                   T5D_OUT_HEADS_VALUE, E, Ep, at, tile, norm, second);
}

extern "C" int t5d_gemm_rows_takes_norm(int K) { return K > 0 && rows_direct(K, K); }

extern "C" int t5d_gemm_rows_normed(void* stream, int w_dtype, const void* A,
                                    const void* W, const float* scales,
                                    const void* residual, void* C, int64_t M, int K,
                                    int N, int epilogue, int out_layout, int E, int Ep,
                                    const int32_t* at, int tile,
                                    const t5d_rows_norm* norm) {
  T5D_REQUIRE(norm, T5D_EINVAL, "t5d_gemm_rows_normed: null pointer");
  T5D_REQUIRE(!at || out_layout == T5D_OUT_HEADS_VALUE, T5D_EINVAL,
              "t5d_gemm_rows_normed: positions go with the value layout");
  return gemm_rows(stream, w_dtype, A, W, scales, residual, C, M, K, N, epilogue,
                   out_layout, E, Ep, at, tile, norm);
}

extern "C" int t5d_gemm_rows_tiled(void* stream, int w_dtype, const void* A,
                                   const void* W, const float* scales,
                                   const void* residual, void* C, int64_t M,
                                   int K, int N, int epilogue, int out_layout,
                                   int E, int Ep, int tile) {
  return gemm_rows(stream, w_dtype, A, W, scales, residual, C, M, K, N, epilogue,
                   out_layout, E, Ep, nullptr, tile);
}

extern "C" int t5d_gemm_rows_values(void* stream, int w_dtype, const void* A,
                                    const void* W, const float* scales, void* C,
                                    int64_t M, int K, int N, const int32_t* at, int E,
                                    int Ep) {
  T5D_REQUIRE(at, T5D_EINVAL, "t5d_gemm_rows_values: null pointer");
  return gemm_rows(stream, w_dtype, A, W, scales, nullptr, C, M, K, N, T5D_EPI_NONE,
                   T5D_OUT_HEADS_VALUE, E, Ep, at, 0);
}

int t5d::launch_dense_rows(hipStream_t s, const void* A, int lda,
                           const void* W, void* C, int out_f32, int ldc,
                           int n_store, int M, int K, int N, int epilogue,
                           float glu_limit, float glu_alpha,
                           float glu_add) {
  RowsGemmArgs g = {};
  g.A = (const bf16_t*)A; g.W = (const char*)W;
  g.scales = nullptr; g.residual = nullptr;
  g.C = out_f32 ? nullptr : (bf16_t*)C;
  g.C32 = out_f32 ? (float*)C : nullptr;
  g.M = M; g.K = K; g.N = N;
  g.epilogue = epilogue; g.layout = T5D_OUT_ROWS;
  g.E = g.Ep = g.H = 0; g.at = nullptr;
  g.lda = lda; g.ldc = ldc; g.n_store = n_store;
  g.gate = tls_gate; g.grp = GroupTiles(); g.n_tiles = 0;
  g.glu_limit = glu_limit; g.glu_alpha = glu_alpha; g.glu_add = glu_add;
  if (g.M <= 128) {  // (float32 results of many columns: see t5d_dense)
    const dim3 grid((g.N + 127) / 128), block(256);
    if (g.M <= 64)
      hipLaunchKernelGGL((rows_gemm_direct_kernel<bf16_t, true, 4, 2, 3, 2, false, true>),
                         grid, block, 0, s, g);
    else
      hipLaunchKernelGGL((rows_gemm_direct_kernel<bf16_t, true, 8, 2, 2, 2, false, true>),
                         grid, block, 0, s, g);
    T5D_CHECK_LAUNCH("t5d_dense(columns)");
    return T5D_OK;
  }
  return launch_rows(s, T5D_BF16, g, 0);
}

int t5d::launch_grouped_rows(hipStream_t s, const GroupedArgs& a, int n_tiles) {
  RowsGemmArgs g = {};
  g.A = a.A; g.W = (const char*)a.W;
  g.scales = nullptr; g.residual = nullptr;
  g.C = (bf16_t*)a.C; g.C32 = nullptr;
  g.M = 0; g.K = a.K; g.N = a.N;
  g.epilogue = a.epilogue; g.layout = T5D_OUT_ROWS;
  g.E = g.Ep = g.H = 0; g.at = nullptr;
  g.lda = a.lda; g.ldc = a.ldc; g.n_store = a.n_store;
  g.glu_limit = a.glu_limit; g.glu_alpha = a.glu_alpha; g.glu_add = a.glu_add;
  g.gate = a.gate; g.grp = a.grp; g.n_tiles = n_tiles;
  // (32 tiles, two workgroups of rows each, make a round over the XCDs)
  const unsigned t64 = (unsigned)(n_tiles + 31) / 32 * 64;
  const unsigned n128 = (g.N + 127) / 128, n256 = (g.N + 255) / 256;
  const bool glu = g.epilogue == T5D_EPI_CLAMPED_GLU;
  // 256 columns unless much of the last column block would be empty
  const bool wide = n256 * 256 <= n128 * 128 + 64;
  const dim3 grid(t64 * (wide ? n256 : n128)), block(256);
  if (wide && glu)
    hipLaunchKernelGGL((rows_gemm_direct_kernel<bf16_t, true, 8, 4, 2, 1, true>), grid, block, 0,
                       s, g);
  else if (wide)
    hipLaunchKernelGGL((rows_gemm_direct_kernel<bf16_t, true, 8, 4, 2, 0, true>), grid, block, 0,
                       s, g);
  else if (glu)
    hipLaunchKernelGGL((rows_gemm_direct_kernel<bf16_t, true, 8, 2, 3, 1, true>), grid, block, 0,
                       s, g);
  else
    hipLaunchKernelGGL((rows_gemm_direct_kernel<bf16_t, true, 8, 2, 3, 0, true>), grid, block, 0,
                       s, g);
  T5D_CHECK_LAUNCH("t5d_grouped_dense_run(rows)");
  return T5D_OK;
}
