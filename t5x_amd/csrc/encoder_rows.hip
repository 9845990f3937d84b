// Which rows an encoder computes.  A batch [B, E] of texts of unequal length holds
// padding after each text, and all padding positions of a text have one and the same
// result: the same embedding goes in, the bias by position drowns in the mask, so each
// attends uniformly over all E positions (t5x/examples/t5/layers.py:309-311,
// network.py:325-328).  So a text of n < E tokens needs n + 1 rows: its own and one of
// padding, which attention counts E - n times (enc_attn_tile_kernel).  Rows of a text
// start at multiples of 4 (what a store of the value layout covers); those in between
// are padding rows too.  The results spread to [B, E] in the final norm
// (t5d_rmsnorm_rows).
// Measured with the dense layers and attention over these rows instead of all
// positions: 12 layers of width 768, 32 texts of 128 to 512 tokens 4.27 -> 3.41 ms; 24
// of width 1024, 7 of 400 to 1031 8.56 -> 6.61 ms.
// The two kernels last 16 us together at 32 x 512 (131 KB of tokens), 14 at 1 x 20 and 23 at
// 1000 x 128, and 3 more where the texts are listed by length.  What bounds them: a launch each, and three atomics of 256 threads on one word
// of LDS each (token_mask_kernel, which reads as much and has one, lasts 4.4 us).
#include "common.h"

namespace t5d {

__device__ __forceinline__ int rows_of_text(int n, int E) {
  return ((n < E ? n + 1 : E) + 3) & ~3;
}

// One workgroup per text: its length, and whether it is tokens followed by zeros.
__global__ void __launch_bounds__(256)
encoder_lengths_kernel(const int64_t* __restrict__ tokens, int32_t* __restrict__ len,
                       int32_t* __restrict__ odd, int E) {
  __shared__ int s_count, s_last, s_other;
  if (threadIdx.x == 0) s_count = s_last = s_other = 0;
  __syncthreads();
  const int64_t* row = tokens + (size_t)blockIdx.x * E;
  int count = 0, last = 0, other = 0;
  for (int e = threadIdx.x; e < E; e += 256) {
    const int64_t t = row[e];
    count += t > 0;
    if (t > 0) last = e + 1;
    other |= t < 0;
  }
  atomicAdd(&s_count, count);
  atomicMax(&s_last, last);
  atomicOr(&s_other, other);
  __syncthreads();
  if (threadIdx.x != 0) return;
  len[blockIdx.x] = s_count;
  odd[blockIdx.x] = s_other | (s_last != s_count);
}

// One workgroup per text: its rows' ids, the row of every position, the position
// (text << 12 | position) of every 4 rows, and (ORDERED) its place by length, for which it
// looks at every text and not only at those before it; the last also sums up for the host.
template <bool ORDERED>
__global__ void __launch_bounds__(256)
encoder_rows_kernel(const int64_t* __restrict__ tokens, const int32_t* __restrict__ len,
                    const int32_t* __restrict__ odd, int32_t* __restrict__ first,
                    int32_t* __restrict__ ids, int32_t* __restrict__ row_of,
                    int32_t* __restrict__ at, int32_t* __restrict__ summary,
                    int32_t* __restrict__ order, int B, int E) {
  __shared__ int s_first, s_most, s_odd, s_longer;
  if (threadIdx.x == 0) s_first = s_most = s_odd = s_longer = 0;
  __syncthreads();
  const int b = blockIdx.x;
  int n = 0;
  if constexpr (ORDERED) n = len[b];
  int before = 0, most = 0, any = 0, longer = 0;
  for (int i = threadIdx.x; i < (ORDERED ? B : b + 1); i += 256) {
    const int other = len[i];
    if constexpr (ORDERED) {
      longer += other > n || (other == n && i < b);
      if (i > b) continue;
    }
    const int rows = rows_of_text(other, E);
    if (i < b) before += rows;
    most = max(most, rows);
    any |= odd[i];
  }
  atomicAdd(&s_first, before);
  atomicMax(&s_most, most);
  atomicOr(&s_odd, any);
  if constexpr (ORDERED) atomicAdd(&s_longer, longer);
  __syncthreads();
  if constexpr (!ORDERED) n = len[b];
  const int r0 = s_first, rows = rows_of_text(n, E);
  if (threadIdx.x == 0) {
    first[b] = r0;
    if constexpr (ORDERED) order[s_longer] = b;
    if (b == B - 1) {
      first[B] = r0 + rows;
      summary[0] = r0 + rows;
      summary[1] = s_most;
      summary[2] = s_odd;
    }
  }
  const int64_t* row = tokens + (size_t)b * E;
  for (int e = threadIdx.x; e < rows; e += 256) {
    ids[r0 + e] = e < n ? (int32_t)row[e] : 0;
    if ((e & 3) == 0) at[(r0 + e) >> 2] = b << 12 | e;
  }
  for (int e = threadIdx.x; e < E; e += 256) row_of[(size_t)b * E + e] = r0 + min(e, n);
}

// One workgroup per text: a bit per position that holds a token, and the last such
// position + 1.
__global__ void __launch_bounds__(256)
token_mask_kernel(const int64_t* __restrict__ tokens, int32_t* __restrict__ last,
                  uint32_t* __restrict__ bits, int E) {
  __shared__ int s_last;
  if (threadIdx.x == 0) s_last = 0;
  __syncthreads();
  const int64_t* row = tokens + (size_t)blockIdx.x * E;
  const int words = (E + 31) >> 5, lane = threadIdx.x & 63;
  int end = 0;
  for (int e0 = 0; e0 < E; e0 += 256) {  // (no lane leaves a wavefront early)
    const int e = e0 + threadIdx.x;
    const bool is = e < E && row[e] > 0;
    const unsigned long long all = __builtin_amdgcn_ballot_w64(is);
    if ((lane & 31) == 0 && (e >> 5) < words)
      bits[(size_t)blockIdx.x * words + (e >> 5)] = (uint32_t)(all >> lane);
    if (is) end = e + 1;
  }
  atomicMax(&s_last, end);
  __syncthreads();
  if (threadIdx.x == 0) last[blockIdx.x] = s_last;
}

}  // namespace t5d

using namespace t5d;

extern "C" int t5d_token_mask(void* stream, const int64_t* tokens, int B, int E,
                              int32_t* last, uint32_t* bits) {
  T5D_REQUIRE(tokens && last && bits, T5D_EINVAL, "t5d_token_mask: null pointer");
  T5D_REQUIRE(B > 0 && E > 0 && E < (1 << 30), T5D_EINVAL, "t5d_token_mask: B=%d E=%d", B,
              E);
  hipLaunchKernelGGL(token_mask_kernel, dim3(B), dim3(256), 0, as_stream(stream), tokens,
                     last, bits, E);
  T5D_CHECK_LAUNCH("t5d_token_mask");
  return T5D_OK;
}

extern "C" int t5d_encoder_rows(void* stream, const int64_t* tokens, int B, int E,
                                int32_t* len, int32_t* odd, int32_t* first,
                                int32_t* ids, int32_t* row_of, int32_t* at,
                                int32_t* summary) {
  return t5d_encoder_rows_ordered(stream, tokens, B, E, len, odd, first, ids, row_of, at,
                                  summary, nullptr);
}

extern "C" int t5d_encoder_rows_ordered(void* stream, const int64_t* tokens, int B, int E,
                                        int32_t* len, int32_t* odd, int32_t* first,
                                        int32_t* ids, int32_t* row_of, int32_t* at,
                                        int32_t* summary, int32_t* order) {
  T5D_REQUIRE(tokens && len && odd && first && ids && row_of && at && summary,
              T5D_EINVAL, "t5d_encoder_rows: null pointer");
  T5D_REQUIRE(B > 0 && E > 0, T5D_EINVAL, "t5d_encoder_rows: B=%d E=%d", B, E);
  T5D_REQUIRE(E <= kMaxEncLen && B < (1 << 19) && (int64_t)B * ((E + 3) / 4 * 4) < (1 << 30),
              T5D_ELIMIT, "t5d_encoder_rows: B=%d E=%d", B, E);
  hipLaunchKernelGGL(encoder_lengths_kernel, dim3(B), dim3(256), 0, as_stream(stream),
                     tokens, len, odd, E);
  if (order)
    hipLaunchKernelGGL(encoder_rows_kernel<true>, dim3(B), dim3(256), 0,
                       as_stream(stream), tokens, len, odd, first, ids, row_of, at,
                       summary, order, B, E);
  else
    hipLaunchKernelGGL(encoder_rows_kernel<false>, dim3(B), dim3(256), 0,
                       as_stream(stream), tokens, len, odd, first, ids, row_of, at,
                       summary, order, B, E);
  T5D_CHECK_LAUNCH("t5d_encoder_rows");
  return T5D_OK;
}
