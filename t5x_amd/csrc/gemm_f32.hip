// Float32 dense layers on the matrix cores (K a multiple of 32, 16-byte rows).
//
// v_mfma_f32_16x16x4_f32 adds its four products to each sum one after the other in
// ascending k, rounding each time, exactly as a chain of fmaf does.  So the sums here
// have the bits of gemm_f32_kernel (gemm.hip), whose order they keep whatever the tile:
// K is cut into 16 contiguous parts of whole 32s; within a part four chains run over
// k % 32 / 8 = 0..3; chains and parts are added in one fixed tree.  A result does not
// depend on the tile or on how many rows a call carries.
//
// What bounds it: a few rows, the stream of weights (a launch holds the whole weight
// tile of its columns in flight); many rows, the float32 matrix rate (157 TFLOP/s) and
// what a CU takes in from its L2.  A wavefront owns whole parts of K, so there is
// nothing to share and no barrier until the one sum at the end: activations are loaded
// 16 bytes per lane and brought into operand order by four lane swaps per 16 k, weights
// 4 to 16 bytes per lane (VW neighbouring columns).
#include "common.h"
#include "gemm_tiles.h"

namespace t5d {

// 4 x 4 transpose between register index and 16-lane row: f[e] of row q becomes
// f[q] of row e.
__device__ __forceinline__ void transpose_rows4(float (&f)[4]) {
  const auto swap32 = [](float& a, float& b) {
    const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(a),
                                                    __float_as_uint(b), false, false);
    a = __uint_as_float(w[0]);
    b = __uint_as_float(w[1]);
  };
  const auto swap16 = [](float& a, float& b) {
    const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(a),
                                                    __float_as_uint(b), false, false);
    a = __uint_as_float(w[0]);
    b = __uint_as_float(w[1]);
  };
  swap32(f[0], f[2]);
  swap32(f[1], f[3]);
  swap16(f[0], f[1]);
  swap16(f[2], f[3]);
}

template <int VW>
__device__ __forceinline__ void load_columns(const float* p, float* v) {
  if constexpr (VW == 4) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  } else {
    v[0] = *p;
  }
}

// A workgroup owns 16 rows and 16 VW output columns; its WV wavefronts (16 or 4)
// take one or four of the 16 parts of K each.  GLU: gated pair (VW values and VW gates
// per lane), plain GELU or, DENSE, the clamped unit.
template <int WV, int VW, bool GLU, bool NORMED, bool DENSE>
__global__ void __launch_bounds__(64 * WV)
gemm_f32_mfma_kernel(F32GemmArgs g) {
  constexpr int NT = GLU ? 2 * VW : VW;
  constexpr int PARTS = 16 / WV;  // of a wavefront
  __shared__ float red[WV][NT * 4][64];
  __shared__ float red_ss[WV][NORMED ? 16 : 1];
  T5D_GATE_READ(g.gate);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int cols = GLU ? g.N >> 1 : g.N;
  const int n0 = blockIdx.x * 16 * VW, m0 = blockIdx.y * 16;
  const int n = min(n0 + c * VW, cols - VW);  // (columns past the edge are not stored)
  const int kq = ((g.K + 15) / 16 + 31) & ~31;

  const float* arow = g.A + (size_t)min(m0 + c, g.M - 1) * g.lda + 4 * q;  // (nor rows)
  const float* wcol = g.W + (size_t)q * g.N + n;

  // What a block of 32 k holds of this lane: activations of k = 16 t + 4 q .., weights
  // of k = 4 j + q.
  struct Block {
    float4 a[2];
    float4 g[NORMED ? 2 : 1];
    float w[8][NT];
  };
  const auto load = [&](Block& b, int k) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      b.a[t] = *reinterpret_cast<const float4*>(arow + k + 16 * t);
    if constexpr (NORMED) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        b.g[t] = *reinterpret_cast<const float4*>(g.norm_scale + k + 16 * t + 4 * q);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float* p = wcol + (size_t)(k + 4 * j) * g.N;
      load_columns<VW>(p, &b.w[j][0]);
      if constexpr (GLU) load_columns<VW>(p + cols, &b.w[j][VW]);
    }
  };

  f32x4_v pair[NT], sum[NT];  // of one part, of up to four
  float pair_ss = 0.f, sum_ss = 0.f;
  Block cur;
  // Part p of this wavefront: with WV = 4 in the order of the tree, i, i + 8, i + 1, i + 9.
  const auto part_of = [&](int p) {
    return WV == 16 ? wave : 2 * wave + (p >> 1) + 8 * (p & 1);
  };
  const auto begin_of = [&](int p) { return min(g.K, part_of(p) * kq); };
  const auto end_of = [&](int p) { return min(g.K, part_of(p) * kq + kq); };
  // parts past the end of K are empty, and so are those behind them that are 8 further
  if (begin_of(0) < g.K) load(cur, begin_of(0));
  T5D_GATE_TEST();
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
    f32x4_v acc[4][NT];
    float ss[2] = {0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[s][nt] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
    const int ke = end_of(p);
    for (int k = begin_of(p); k < ke; k += 32) {
      Block b = cur;
      // the block after this one: of this part, of the next, or of the one behind an
      // empty one
      int next = k + 32;
      if (next >= ke) {
        next = p + 1 < PARTS ? begin_of(p + 1) : g.K;
        if (next >= g.K && p + 2 < PARTS) next = begin_of(p + 2);
      }
      if (next < g.K) load(cur, next);
      if constexpr (NORMED) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          float s[4] = {b.g[t].x, b.g[t].y, b.g[t].z, b.g[t].w};
          transpose_rows4(s);
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) b.w[4 * t + j][nt] *= s[j];
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float a[4] = {b.a[t].x, b.a[t].y, b.a[t].z, b.a[t].w};
        if constexpr (NORMED) {
          // the chain of 8 k runs through an even and then an odd row of lanes
          float x = ss[t];
#pragma unroll
          for (int e = 0; e < 4; ++e) x = fmaf(a[e], a[e], x);
          auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(x),
                                                    __float_as_uint(x), false, false);
          x = __uint_as_float(w[0]);
#pragma unroll
          for (int e = 0; e < 4; ++e) x = fmaf(a[e], a[e], x);
          w = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x),
                                               false, false);
          ss[t] = __uint_as_float(w[1]);
        }
        transpose_rows4(a);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            f32x4_v& x = acc[2 * t + (j >> 1)][nt];
            x = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b.w[4 * t + j][nt], x, 0, 0, 0);
          }
      }
    }
    // the tree: chains of the part, then parts i and i + 8, then pairs of those
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const f32x4_v s = (acc[0][nt] + acc[1][nt]) + (acc[2][nt] + acc[3][nt]);
      if (p == 0) sum[nt] = s;
      else if (p == 1) sum[nt] += s;
      else if (p == 2) pair[nt] = s;
      else sum[nt] += pair[nt] + s;
    }
    if constexpr (NORMED) {
      const auto halves = [](float x) {
        const auto w = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(x), __float_as_uint(x), false, false);
        return __uint_as_float(w[0]) + __uint_as_float(w[1]);
      };
      const float s = halves(ss[0]) + halves(ss[1]);
      if (p == 0) sum_ss = s;
      else if (p == 1) sum_ss += s;
      else if (p == 2) pair_ss = s;
      else sum_ss += pair_ss + s;
    }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][nt * 4 + i][lane] = sum[nt][i];
  if (NORMED && q == 0) red_ss[wave][c] = sum_ss;
  __syncthreads();
  const auto tree = [](const auto& part) {
    if constexpr (WV == 4)
      return (part(0) + part(1)) + (part(2) + part(3));
    else {
      const auto r = [&](int i) { return part(i) + part(i + 8); };
      return ((r(0) + r(1)) + (r(2) + r(3))) + ((r(4) + r(5)) + (r(6) + r(7)));
    }
  };
  for (int e = threadIdx.x; e < 16 * 16 * VW; e += 64 * WV) {
    const int ml = e / (16 * VW), l = e % (16 * VW);
    const int row = m0 + ml, col = n0 + l;
    if (row >= g.M || col >= cols) continue;
    const int at = (ml >> 2) * 16 + l / VW;
    const auto total = [&](int nt) {
      return tree([&](int w) { return red[w][nt * 4 + (ml & 3)][at]; });
    };
    float inv = 1.f;
    if constexpr (NORMED)
      inv = 1.0f / sqrtf(tree([&](int w) { return red_ss[w][ml]; }) / (float)g.K + g.eps);
    float v = total(l % VW) * inv;
    if constexpr (GLU) {
      const float vg = total(VW + l % VW) * inv;
      v = DENSE ? clamped_glu(v, vg, g.glu_limit, g.glu_alpha, g.glu_add)
                : gelu_tanh(v) * vg;
    } else if (g.epilogue == T5D_EPI_RESIDUAL) {
      v += g.residual[(size_t)row * g.N + col];
    }
    g.C[(size_t)row * cols + col] = v;
  }
}

// Few workgroups take 16 wavefronts, a part of K each, so that a CU has the whole tile
// in flight; once they are more than the chip holds at a time (two per CU), four
// wavefronts and, without a gate, 64 columns read less per product.  Measured, us before
// (8 rows x 16 columns, vector units) / 16 wavefronts x 16 columns / 4 x 16 / 4 x 64:
//   8 x 512 x 1152 normed        6.5 /   4.0 /   4.5 /  8.2     (72 workgroups)
//   8 x 1024 x 512 residual      7.9 /   4.4 /   5.1 /  9.5
//   100 x 512 x 2048 gated      23.9 /   9.6 /   9.6 /   -      (448)
//   512 x 512 x 1152 normed    100.9 /  26.3 /  20.5 / 19.5     (2304)
//   512 x 512 x 2048 gated      90.5 /  33.3 /  26.4 /   -
//   2000 x 1024 x 512          229.4 /  47.6 /  44.9 / 36.3
//   8 x 512 x 32128             41.8 /  20.4 /  20.6 / 13.3     (5.0 TB/s)
template <bool GLU, bool NORMED, bool DENSE>
static void launch_f32_tile(hipStream_t s, const F32GemmArgs& g) {
  const int cols = GLU ? g.N >> 1 : g.N;
  const unsigned m_tiles = (g.M + 15) / 16;
  const dim3 grid((cols + 15) / 16, m_tiles);
  if ((int64_t)grid.x * grid.y <= 512) {
    hipLaunchKernelGGL((gemm_f32_mfma_kernel<16, 1, GLU, NORMED, DENSE>), grid,
                       dim3(1024), 0, s, g);
    return;
  }
  if constexpr (!GLU) {
    if (cols % 4 == 0 && ((uintptr_t)g.W & 15) == 0) {
      hipLaunchKernelGGL((gemm_f32_mfma_kernel<4, 4, GLU, NORMED, DENSE>),
                         dim3((cols + 63) / 64, m_tiles), dim3(256), 0, s, g);
      return;
    }
  }
  hipLaunchKernelGGL((gemm_f32_mfma_kernel<4, 1, GLU, NORMED, DENSE>), grid,
                     dim3(256), 0, s, g);
}

bool launch_f32_mfma(hipStream_t s, const F32GemmArgs& g, bool dense) {
  if (g.K % 32 != 0 || g.K < 128 || g.lda % 4 != 0 || ((uintptr_t)g.A & 15) != 0 ||
      ((uintptr_t)g.norm_scale & 15) != 0)
    return false;
  if (dense) {
    if (g.epilogue == T5D_EPI_CLAMPED_GLU) launch_f32_tile<true, false, true>(s, g);
    else launch_f32_tile<false, false, true>(s, g);
  } else if (g.norm_scale != nullptr) {
    if (g.epilogue == T5D_EPI_GEGLU) launch_f32_tile<true, true, false>(s, g);
    else launch_f32_tile<false, true, false>(s, g);
  } else {
    if (g.epilogue == T5D_EPI_GEGLU) launch_f32_tile<true, false, false>(s, g);
    else launch_f32_tile<false, false, false>(s, g);
  }
  return true;
}

}  // namespace t5d
