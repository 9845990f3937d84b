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

template <typename Args> struct IsStream { static constexpr bool value = false; };
template <> struct IsStream<StreamDenseArgs> { static constexpr bool value = true; };
__device__ __forceinline__ int columns_of_norm(const GemmArgs& g) { return g.K; }
__device__ __forceinline__ int columns_of_norm(const StreamDenseArgs& g) { return g.d; }
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

// norm_dense_kernel; false where norm_gemm_kernel is faster, nothing is launched then.
bool launch_norm_dense(int w_dtype, const GemmArgs& g, hipStream_t s);

// The arguments of t5d_stream_dense and t5d_stream_rows_dense, checked (stream_dense.hip).
int stream_dense_args(const char* name, StreamDenseArgs* g, int most_rows, const void* y,
                      const float* y_norm, const float* x, float* x_out, const float* norm,
                      int d, float eps, const void* W, int out_dtype, void* C, int ldc,
                      int n_store, int M, int ld, int N, int epilogue, float glu_limit,
                      float glu_alpha, float glu_add);

}  // namespace t5d
#endif  // T5D_NORM_DENSE_H_
