// A norm and the dense layer behind it in one launch: arguments of the two kernels.
#ifndef T5D_NORM_DENSE_H_
#define T5D_NORM_DENSE_H_
#include "common.h"
#include "gemm_tiles.h"

namespace t5d {

// The row kernel of a float32 stream (t5d_stream_norm) and the layer behind it.
struct StreamDenseArgs : DenseArgs {
  const bf16_t* y;                  // [M, lda] branch output, or null
  const float *y_norm, *x, *norm;   // [d] or null; [M, lda]; [d]
  float* x_out;                     // [M, lda], not x: the stream with the branch added
  int d;
};

// The norms of the new latents (latent_append_kernel) and the layer behind the queries'.
struct LatentDenseArgs : DenseArgs {
  const float* norm;     // [K], zeros behind the d of the latent; A's rows: lda apart
  int d;
  // The cached latents' norm and way into the ring, by workgroups of their own behind the
  // first dense_blocks; kv null: none.
  int dense_blocks;
  const bf16_t* kv;      // [M, ..], rows lda apart
  const float* kv_norm;  // [kv_pad]
  int kv_d, kv_pad, ring_len;
  bf16_t* ring;          // [slots, ring_len, kv_pad]
  const int32_t *seq_slot, *tok_seq, *tok_pos;
};

template <typename Args> struct IsLatent { static constexpr bool value = false; };
template <> struct IsLatent<LatentDenseArgs> { static constexpr bool value = true; };
template <typename Args> struct IsStream { static constexpr bool value = false; };
template <> struct IsStream<StreamDenseArgs> { static constexpr bool value = true; };
__device__ __forceinline__ int columns_of_norm(const GemmArgs& g) { return g.K; }
__device__ __forceinline__ int columns_of_norm(const StreamDenseArgs& g) { return g.d; }
__device__ __forceinline__ int columns_of_norm(const LatentDenseArgs& g) { return g.K; }
__device__ __forceinline__ int d_of_norm(const GemmArgs& g) { return g.K; }
__device__ __forceinline__ int d_of_norm(const LatentDenseArgs& g) { return g.d; }
__device__ __forceinline__ bool has_branch(const GemmArgs&) { return false; }
__device__ __forceinline__ bool has_branch(const StreamDenseArgs& g) {
  return g.y != nullptr;
}
__device__ __forceinline__ float4 norm_column(const float* p, int c, int d) {
  float4 w = make_float4(0.f, 0.f, 0.f, 0.f);  // 4 entries of a [d] vector
  if (c + 4 <= d) return *reinterpret_cast<const float4*>(p + c);
  if (c < d) w.x = p[c];
  if (c + 1 < d) w.y = p[c + 1];
  if (c + 2 < d) w.z = p[c + 2];
  return w;
}

// 8 columns from c on of a latent's row of `have` columns, and the same normed.
__device__ __forceinline__ uint4 latent_piece(const bf16_t* row, int c, int have) {
  return c < have ? *reinterpret_cast<const uint4*>(row + c) : make_uint4(0, 0, 0, 0);
}
__device__ __forceinline__ uint4 latent_normed(const uint4& x, float inv, const float* w) {
  float f[8];
  unpack16(x, f);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = f[e] * inv * w[e];
  return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]),
                    pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
}

// norm_dense_kernel; false where norm_gemm_kernel is faster, nothing is launched then.
bool launch_norm_dense(int w_dtype, const GemmArgs& g, hipStream_t s);
// The same for the latents of a step; false: two kernels instead.
bool launch_latent_dense(LatentDenseArgs g, hipStream_t s);

// The arguments of t5d_stream_dense and t5d_stream_rows_dense, checked (stream_dense.hip).
int stream_dense_args(const char* name, StreamDenseArgs* g, int most_rows, const void* y,
                      const float* y_norm, const float* x, float* x_out, const float* norm,
                      int d, float eps, const void* W, int out_dtype, void* C, int ldc,
                      int n_store, int M, int ld, int N, int epilogue, float glu_limit,
                      float glu_alpha, float glu_add);

}  // namespace t5d
#endif  // T5D_NORM_DENSE_H_
