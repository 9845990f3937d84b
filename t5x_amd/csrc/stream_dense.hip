// The row kernel between two dense layers (t5d_stream_norm) and the layer behind it in one
// launch, for a few rows: every workgroup forms the rows it multiplies by itself.
#include "common.h"
#include "gemm_tiles.h"
#include "norm_dense.h"

namespace t5d {

// Rows x + norm(y) and their norm as t5d_stream_norm forms them, then 16 NT columns of the
// layer as gemm_mfma_kernel does: the same bits as the two of them.  256 threads hold RM
// rows in VPT groups of 4 columns; the normed rows meet the matrix cores through LDS; K is
// cut into pairs of k-tiles over the 4 wavefronts, NJ at most each, all of whose weights are
// requested behind the rows and arrive while these are normed.  The first workgroup stores
// the stream, into another buffer than the one that the others may still be reading.
// What bounds it: the chain launch, rows, two sums over the workgroup, products, sum over
// the wavefronts, in the place of two such chains; with more rows what every workgroup
// fetches and norms anew, hence up to 4.  us, weights from memory, the two kernels / this one:
//   rows                         1            2            4            8
//   1024 x 3328             6.3 /  3.5   6.4 /  4.0   6.5 /  5.0   6.6 /  6.9
//   1024 x 5632 gated       7.7 /  4.6   7.6 /  5.4   7.7 /  6.8   8.0 /  9.3
//   1024 x 32128 float32   17.2 / 13.4  17.0 / 14.4  17.1 / 15.5  17.5 / 19.1
//   768 x 4096 gated        6.1 /  3.5   6.3 /  4.0   6.4 /  5.0   6.6 /  6.9
//   2048 x 10240 gated     15.0 / 11.5  15.0 / 12.2  14.7 / 13.3  14.9 / 21.7
// A step of one row, 8 layers of width 1024: 284 -> 228 us.
template <int RM, int NT, int NJ, int VPT>
__global__ void __launch_bounds__(256)
stream_dense_kernel(StreamDenseArgs g) {
  constexpr int TN = 16 * NT, LD = 1024 * VPT;
  constexpr int HS = LD + 8;  // row stride of the normed rows
  __shared__ float s_sum[2][RM][4];
  __shared__ __align__(16) bf16_t s_h[RM * HS];
  __shared__ float red[4][NT * 4][64];
  T5D_GATE_READ(g.gate);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ld = g.lda, KT = ld >> 5, n_pairs = KT >> 1;
  const int n_tiles_total = g.N >> 4, nt0 = blockIdx.x * NT;

  float4 x[RM][VPT];
  uint2 y[RM][VPT];
  bool on[VPT];
#pragma unroll
  for (int v = 0; v < VPT; ++v) on[v] = 4 * ((int)threadIdx.x + 256 * v) < ld;
#pragma unroll
  for (int r = 0; r < RM; ++r) {
    const size_t row = (size_t)min(r, g.M - 1) * ld;  // (past the end: not stored)
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      const int c = 4 * (threadIdx.x + 256 * v);
      x[r][v] = on[v] ? *reinterpret_cast<const float4*>(g.x + row + c)
                      : make_float4(0.f, 0.f, 0.f, 0.f);
      y[r][v] = on[v] && g.y != nullptr ? *reinterpret_cast<const uint2*>(g.y + row + c)
                                        : make_uint2(0, 0);
    }
  }
  float4 wy[VPT], wx[VPT];
#pragma unroll
  for (int v = 0; v < VPT; ++v) {
    const int c = 4 * (threadIdx.x + 256 * v);
    wy[v] = g.y_norm != nullptr ? norm_column(g.y_norm, c, g.d) : make_float4(1.f, 1.f, 1.f, 1.f);
    wx[v] = norm_column(g.norm, c, g.d);
  }
  uint4 w[NJ][2][NT];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int nn = 0; nn < NT; ++nn)
        w[j][h][nn] = WeightTile<bf16_t>::load(
            reinterpret_cast<const char*>(g.W) +
                ((size_t)min(nt0 + nn, n_tiles_total - 1) * KT +
                 2 * min(wave + 4 * j, n_pairs - 1) + h) * 1024,
            lane);
  T5D_GATE_TEST();

  // sums over the workgroup of one value per row
  const auto block_sums = [&](float (&v)[RM], float (*s)[4]) {
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      v[r] = wave_sum(v[r]);
      if (lane == 0) s[r][wave] = v[r];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (what is requested comes later)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < RM; ++r) v[r] = (s[r][0] + s[r][1]) + (s[r][2] + s[r][3]);
  };
  float ss[RM];
  if (g.y != nullptr) {
    const bool normed = g.y_norm != nullptr;
    if (normed) {
#pragma unroll
      for (int r = 0; r < RM; ++r) {
        ss[r] = 0.f;
#pragma unroll
        for (int v = 0; v < VPT; ++v) {
          const float y0 = bf16lo_to_f32(y[r][v].x), y1 = bf16hi_to_f32(y[r][v].x);
          const float y2 = bf16lo_to_f32(y[r][v].y), y3 = bf16hi_to_f32(y[r][v].y);
          ss[r] = fmaf(y0, y0, ss[r]); ss[r] = fmaf(y1, y1, ss[r]);
          ss[r] = fmaf(y2, y2, ss[r]); ss[r] = fmaf(y3, y3, ss[r]);
        }
      }
      block_sums(ss, s_sum[0]);
    }
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      const float inv = normed ? 1.0f / sqrtf(ss[r] / (float)g.d + g.eps) : 1.f;
#pragma unroll
      for (int v = 0; v < VPT; ++v) {
        x[r][v].x += bf16lo_to_f32(y[r][v].x) * inv * wy[v].x;
        x[r][v].y += bf16hi_to_f32(y[r][v].x) * inv * wy[v].y;
        x[r][v].z += bf16lo_to_f32(y[r][v].y) * inv * wy[v].z;
        x[r][v].w += bf16hi_to_f32(y[r][v].y) * inv * wy[v].w;
        if (blockIdx.x == 0 && r < g.M && on[v])
          *reinterpret_cast<float4*>(g.x_out + (size_t)r * ld +
                                     4 * (threadIdx.x + 256 * v)) = x[r][v];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RM; ++r) {
    ss[r] = 0.f;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      ss[r] = fmaf(x[r][v].x, x[r][v].x, ss[r]);
      ss[r] = fmaf(x[r][v].y, x[r][v].y, ss[r]);
      ss[r] = fmaf(x[r][v].z, x[r][v].z, ss[r]);
      ss[r] = fmaf(x[r][v].w, x[r][v].w, ss[r]);
    }
  }
  block_sums(ss, s_sum[1]);
#pragma unroll
  for (int r = 0; r < RM; ++r) {
    const float inv = 1.0f / sqrtf(ss[r] / (float)g.d + g.eps);
#pragma unroll
    for (int v = 0; v < VPT; ++v)
      if (on[v])
        *reinterpret_cast<uint2*>(s_h + r * HS + 4 * (threadIdx.x + 256 * v)) = make_uint2(
            pack_bf16x2(x[r][v].x * inv * wx[v].x, x[r][v].y * inv * wx[v].y),
            pack_bf16x2(x[r][v].z * inv * wx[v].z, x[r][v].w * inv * wx[v].w));
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  f32x4_v acc[NT];
#pragma unroll
  for (int nn = 0; nn < NT; ++nn) acc[nn] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  // (rows past RM: any row, columns of the products that nothing looks at)
  const bf16_t* a_from = s_h + (lane & (RM - 1)) * HS + 8 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int pair = wave + 4 * j;
    if (pair >= n_pairs) break;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      Frag a;
      a.u = *reinterpret_cast<const uint4*>(a_from + 64 * pair + 32 * h);
#pragma unroll
      for (int nn = 0; nn < NT; ++nn)
        acc[nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a.v, WeightTile<bf16_t>::frag(w[j][h][nn]).v, acc[nn], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][t * 4 + i][lane] = acc[t][i];
  __syncthreads();
  const bool pair = gated(g);
  const auto tile_sum = [&](int ml, int nl) -> float {
    const int l = (ml >> 2) * 16 + (nl & 15), idx = (nl >> 4) * 4 + (ml & 3);
    return (red[0][idx][l] + red[2][idx][l]) + (red[1][idx][l] + red[3][idx][l]);
  };
#pragma unroll
  for (int e = threadIdx.x; e < RM * TN; e += 256) {
    const int ml = e / TN, nl = e % TN, n = nt0 * 16 + nl;
    if (ml >= g.M || n >= stored_columns(g) || (pair && (nl & 8))) continue;
    store_result(g, ml, n, tile_sum(ml, nl), pair ? tile_sum(ml, nl + 8) : 0.f, 0.f);
  }
}

}  // namespace t5d

using namespace t5d;

extern "C" int t5d_stream_dense_rows(int dtype, int ld) {
  return dtype == T5D_BF16 && ld > 0 && ld % 64 == 0 && ld <= 2048 ? 4 : 0;
}

// Where the many workgroups of a wide layer cost more than the launch they save: each forms
// the rows anew, for few weights where ld is small, and where ld is just above 1024 with
// requests for the pairs of 2048.  us, the two kernels / this one, float32 results (rows x ld
// x columns):
//   4 x   64 x  4096   4.67 /  4.54    4 x   64 x 32128   5.79 /  6.99
//   4 x  128 x  8192   5.44 /  5.36    4 x  128 x 32128   6.41 /  6.97
//   4 x  256 x 32128   8.24 /  7.61    4 x  256 x 50304  10.6 /  11.0
//   4 x  384 x 24576   8.66 /  8.28    4 x  384 x 32128   9.59 / 10.01
//   4 x 1152 x 16384   13.4 /  11.9    4 x 1152 x 32128   19.2 /  20.0
//   4 x 1408 x 16384   14.9 /  13.5    4 x 1408 x 24576   18.2 /  18.7
//   2 x 1088 x 32128   18.8 /  18.3    2 x 1088 x 50304   27.3 /  28.2
//   1 x 1088 x 50304   27.6 /  26.6    1 x 1088 x 131072  54.5 /  57.3
//   2 x  128 x 50304   8.89 /  7.72    2 x  128 x 131072  13.2 /  14.0
//   4 x  512 x 131072  29.7 /  26.9    4 x 1536 x 131072  75.1 /  73.2
//   4 x 1024 x 131072  51.1 /  45.9    4 x 2048 x 131072  95.6 /  86.1
extern "C" int t5d_stream_dense_pays(int M, int ld, int N) {
  const bool between = ld > 1024 && ld < (M >= 3 ? 1536 : 1280);
  if (M >= 3 && ld < 512) return N <= (ld % 256 == 0 ? 128 : 64) * ld;
  if (between) return N <= (M == 1 ? 98304 : M == 2 ? 40960 : 20480);
  return M == 1 || ld >= 256 || N <= 98304;
}

int t5d::stream_dense_args(const char* name, StreamDenseArgs* g, int most_rows, const void* y,
                           const float* y_norm, const float* x, float* x_out,
                           const float* norm, int d, float eps, const void* W, int out_dtype,
                           void* C, int ldc, int n_store, int M, int ld, int N, int epilogue,
                           float glu_limit, float glu_alpha, float glu_add) {
  T5D_REQUIRE(x && norm && W && C && (!y || (x_out && x_out != x)), T5D_EINVAL,
              "%s: null pointer, or the stream in place", name);
  T5D_REQUIRE(M > 0 && M <= most_rows && d > 0 && d <= ld, T5D_ELIMIT,
              "%s: M=%d d=%d ld=%d", name, M, d, ld);
  const bool glu = epilogue == T5D_EPI_CLAMPED_GLU;
  T5D_REQUIRE((epilogue == T5D_EPI_NONE || glu) && N > 0 && N % 16 == 0 &&
                  (out_dtype == T5D_F32
                       ? !glu && n_store > 0 && n_store <= N && ldc >= n_store
                       : out_dtype == T5D_BF16 &&
                             (glu ? ldc == N / 2 && n_store == N
                                  : ldc == N && n_store == N)),
              T5D_EINVAL, "%s: out_dtype %d with epilogue %d, N=%d ldc=%d n_store=%d", name,
              out_dtype, epilogue, N, ldc, n_store);
  T5D_REQUIRE((((uintptr_t)y | (uintptr_t)x | (uintptr_t)x_out | (uintptr_t)W |
                (uintptr_t)C | (uintptr_t)norm | (uintptr_t)y_norm) % 16) == 0,
              T5D_EINVAL, "%s: operands must be 16-byte aligned", name);
  g->A = nullptr; g->W = W; g->scales = nullptr; g->residual = nullptr;
  g->C = C; g->M = M; g->K = ld; g->N = N; g->m_parts = 1;
  g->gate = tls_gate; g->epilogue = epilogue; g->out_f32 = out_dtype == T5D_F32;
  g->norm_scale = nullptr; g->eps = eps;
  g->lda = ld; g->ldc = ldc; g->n_store = n_store;
  g->glu_limit = glu_limit; g->glu_alpha = glu_alpha; g->glu_add = glu_add;
  g->y = (const bf16_t*)y; g->y_norm = y_norm; g->x = x; g->norm = norm;
  g->x_out = x_out; g->d = d;
  return T5D_OK;
}

extern "C" int t5d_stream_dense(void* stream, const void* y, const float* y_norm,
                                const float* x, float* x_out, const float* norm, int d,
                                float eps, const void* W, int out_dtype, void* C, int ldc,
                                int n_store, int M, int ld, int N, int epilogue,
                                float glu_limit, float glu_alpha, float glu_add) {
  StreamDenseArgs g;
  const int rc = stream_dense_args("t5d_stream_dense", &g,
                                   t5d_stream_dense_rows(T5D_BF16, ld), y, y_norm, x, x_out,
                                   norm, d, eps, W, out_dtype, C, ldc, n_store, M, ld, N,
                                   epilogue, glu_limit, glu_alpha, glu_add);
  if (rc != T5D_OK) return rc;
  const int tiles = N / 16;
  const int nt = tiles > 512 ? 2 : 1;
  const dim3 grid((tiles + nt - 1) / nt), block(256);
  hipStream_t s = as_stream(stream);
#define T5D_SD(RM_, NT_, NJ_, VPT_) \
  hipLaunchKernelGGL((stream_dense_kernel<RM_, NT_, NJ_, VPT_>), grid, block, 0, s, g)
#define T5D_SD_K(RM_, NT_)                      \
  do {                                          \
    if (ld <= 512) T5D_SD(RM_, NT_, 2, 1);      \
    else if (ld <= 768) T5D_SD(RM_, NT_, 3, 1); \
    else if (ld <= 1024) T5D_SD(RM_, NT_, 4, 1); \
    else T5D_SD(RM_, NT_, 8, 2);                \
  } while (0)
#define T5D_SD_M(NT_)                           \
  do {                                          \
    if (M == 1) T5D_SD_K(1, NT_);               \
    else if (M == 2) T5D_SD_K(2, NT_);          \
    else T5D_SD_K(4, NT_);                      \
  } while (0)
  if (nt == 1) T5D_SD_M(1);
  else T5D_SD_M(2);
#undef T5D_SD_M
#undef T5D_SD_K
#undef T5D_SD
  T5D_CHECK_LAUNCH("t5d_stream_dense");
  return T5D_OK;
}
