// Single-query ("decode step") attention in float32 — the dtype of exactness tests and
// of users without bfloat16 checkpoints — and what the bfloat16 kernels
// (attention_mfma.hip) share with it.
#include <math.h>

#include "common.h"

namespace t5d {

struct AttnArgs {
  const void* q;        // self: qkv [R, 3*HD]; cross: q [R, HD]
  void* k;              // [G, H, 64, S]
  void* v;              // [G, H, 64, S]
  const void* rel_bias; // self: [H, S] by distance; cross: null
  const int32_t* index; // self: cache_index scalar; cross: enc_len [G]
  void* out;            // [R, HD]
  int H, S, nq, q_stride;
  const int32_t* gate;  // optional device-side enable flag
  // float32: the first wavefront asks for its keys and values before it knows how many
  // positions are valid.  Set while workgroups are few (one per CU): the wait for the
  // length then costs more than requests for positions that turn out to be masked.  With
  // many the traffic does (64 items of 12 heads, 64 positions, 10 valid: 4.3 us, all
  // asked for 6.6).
  bool early;
};

constexpr int kD = 64;
constexpr int kMaxWaves = 16;

// ---- float32 self-attention ----------------------------------------------------
// K and V [R, heads, 64, len] with `len` contiguous — the reference's cache layout
// (t5x/examples/t5/layers.py:226-241).  A workgroup takes one (row, head), wavefront w
// key positions 64 w .. 64 w + 63; inside a wavefront lane = (dg, jc): jc = lane % 16
// selects 4 consecutive positions, dg = lane / 16 head-dim rows d = dg + 4 i, so every
// load fetches 4 rows x 256 contiguous bytes.  Scores are sums over a lane's 16 rows,
// then over dg; maximum and sum of the softmax go over jc (and over wavefronts through
// LDS); weights are normalised before the value product, whose sums over jc end
// scattered: lane (dg, jc) holds d = dg + 4 jc.
//
// What bounds it at the few rows it is used for is a chain of waits and the fetch of
// its own code, whose every KB costs 0.2 us while it is cold.  So everything is asked
// for at the start: new key and value and bias with the queries, the first
// wavefront's keys and values before it knows how many positions are valid (see
// AttnArgs::early); and the new column has a score and a weight of its own: merged into
// the others by 32 branches of the lane that has it, with a comparison per element, the
// kernel had 3456 instructions.  us, before / now: 8 rows of 6 heads over 32 positions
// 8.4 / 3.5, 16 x 12 over 128 9.8 / 5.3, 16 x 6 over 256 10.4 / 5.8, 64 x 12 over 64
// 11.3 / 6.3, 8 x 6 over 1000 20.3 / 12.4.  Error against float64 as before (1.8e-7 over
// 32 positions, 3.4e-7 over 1000).
//
// WM = the most wavefronts a launch of this instance uses; it bounds the
// workgroup size so short key axes get the full register file.
constexpr int kDppRotate8 = 0x128;  // lane i <-> (i + 8) % 16
// One step of the scatter: ST of the 2 ST sums stay, the partner (CTRL: a lane that
// differs in bit ST) adds its own.
template <int ST, int CTRL>
__device__ __forceinline__ void scatter_step(float (&o)[16], int jc) {
  const bool up = (jc & ST) != 0;
#pragma unroll
  for (int k = 0; k < ST; ++k) {
    const float mine = up ? o[k + ST] : o[k];
    const float other = up ? o[k] : o[k + ST];
    o[k] = mine + dpp_move<CTRL>(other);
  }
}

template <int WM>
__global__ void __launch_bounds__(64 * WM)
self_attn_f32_kernel(AttnArgs a) {
  __shared__ float s_red[2][WM];
  __shared__ float s_out[WM][kD];
  T5D_GATE_READ(a.gate);
  const int h = blockIdx.x, g = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nwaves = blockDim.x >> 6;
  const int jc = lane & 15, dg = lane >> 4;
  const int HD = a.H * kD;
  const int j0 = wave * 64 + jc * 4;
  // the cache of this row and head, and this lane's corner of it: row dg, position j0;
  // its rows are 4 S floats apart
  const size_t first = ((size_t)g * a.H + h) * kD * a.S;
  const unsigned corner = dg * a.S + j0;
  const int step = 4 * a.S;
  float* kp = reinterpret_cast<float*>(a.k) + first;
  float* vp = reinterpret_cast<float*>(a.v) + first;
  const float* q = reinterpret_cast<const float*>(a.q) + (size_t)g * a.q_stride +
                   h * kD + dg;
  // (with 16 wavefronts there are no registers for values beside keys)
  constexpr bool kAhead = WM < 16;
  const bool early = kAhead && a.early && wave == 0;

  float qv[16], knew[16], vnew[16];
  const auto request_new = [&](float (&to)[16], int at) {
#pragma unroll
    for (int i = 0; i < 16; ++i) to[i] = q[at + 4 * i];
  };
  request_new(qv, 0);
  request_new(knew, HD);
  if (kAhead) request_new(vnew, 2 * HD);
  float4 kc[16], vc[16];
  const auto request = [&](float4 (&to)[16], const float* from) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      to[i] = *reinterpret_cast<const float4*>(from + i * step + corner);
  };
  if (early && j0 < a.S) {
    request(kc, kp);
    request(vc, vp);
  }

  // A cache index outside [0, S) (a decode loop longer than its cache) must
  // not become an address: nothing is inserted then and all S columns are
  // attended with the bias row of the last position, which is what the
  // reference's one-hot insert and clamped slices do (layers.py:258-303).
  int t = *a.index;
  T5D_GATE_TEST();
  const bool past_end = t < 0 || t >= a.S;
  if (past_end) t = a.S - 1;
  const int n = t + 1;
  const bool live = j0 < n;
  float bias[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    bias[e] = reinterpret_cast<const float*>(a.rel_bias)[(size_t)h * a.S +
                                                         max(t - j0 - e, 0)];
  if (!early && live) {
    request(kc, kp);
    if (kAhead) request(vc, vp);
  }
  // The lane whose positions contain column t takes the new key and value there, whose
  // score is formed beside the others, and writes them to the cache.
  const bool ins = !past_end && t >= j0 && t < j0 + 4;
  float s_new = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) s_new = fmaf(qv[i], knew[i], s_new);
  if (ins) {
    const unsigned col = dg * a.S + t;
#pragma unroll
    for (int i = 0; i < 16; ++i) *(kp + i * step + col) = knew[i];
  }
  if (!kAhead) __builtin_amdgcn_sched_barrier(0);  // (the new key's registers)

  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    s[0] = fmaf(qv[i], kc[i].x, s[0]);
    s[1] = fmaf(qv[i], kc[i].y, s[1]);
    s[2] = fmaf(qv[i], kc[i].z, s[2]);
    s[3] = fmaf(qv[i], kc[i].w, s[3]);
  }
  if (!kAhead) {
    __builtin_amdgcn_sched_barrier(0);  // (the keys' registers)
    if (live) request(vc, vp);
    request_new(vnew, 2 * HD);
  }

  float mx = -INFINITY;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (ins && j0 + e == t) s[e] = s_new;
    s[e] = j0 + e < n ? rows_sum(s[e]) + bias[e] : -INFINITY;
    mx = fmaxf(mx, s[e]);
  }
  mx = lanes16_max(mx);
  if (nwaves > 1) {
    if (lane == 0) s_red[0][wave] = mx;
    __syncthreads();
    mx = s_red[0][0];
    for (int w = 1; w < nwaves; ++w) mx = fmaxf(mx, s_red[0][w]);
  }
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s[e] = s[e] == -INFINITY ? 0.f : expf(s[e] - mx);
    sum += s[e];
  }
  sum = lanes16_sum(sum);
  if (nwaves > 1) {
    if (lane == 0) s_red[1][wave] = sum;
    __syncthreads();
    sum = s_red[1][0];
    for (int w = 1; w < nwaves; ++w) sum += s_red[1][w];
  }
  // A zero weight must not pick up whatever lies past the prefix, nor the new column
  // what its place held.
  uint32_t there[4];
  float p_new = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s[e] /= sum;
    const bool fresh = ins && j0 + e == t;
    if (fresh) p_new = s[e];
    there[e] = s[e] != 0.f && !fresh ? 0xffffffffu : 0u;
    s[e] = fresh ? 0.f : s[e];
  }
  const uint32_t there_new = p_new != 0.f ? 0xffffffffu : 0u;
  const auto masked = [](uint32_t mask, float v) {
    return __uint_as_float(mask & __float_as_uint(v));
  };

  float o[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    o[i] = s[0] * masked(there[0], vc[i].x);
    o[i] = fmaf(s[1], masked(there[1], vc[i].y), o[i]);
    o[i] = fmaf(s[2], masked(there[2], vc[i].z), o[i]);
    o[i] = fmaf(s[3], masked(there[3], vc[i].w), o[i]);
    o[i] = fmaf(p_new, masked(there_new, vnew[i]), o[i]);
  }
  if (ins) {
    const unsigned col = dg * a.S + t;
#pragma unroll
    for (int i = 0; i < 16; ++i) *(vp + i * step + col) = vnew[i];
  }
  // Partners of the scatter: 8 lanes on, mirrored in 8, 2 on, 1 on (each differs in
  // the step's bit; together they are all 16).
  scatter_step<8, kDppRotate8>(o, jc);
  scatter_step<4, kDppHalfMirror>(o, jc);
  scatter_step<2, kDppXor2>(o, jc);
  scatter_step<1, kDppXor1>(o, jc);
  float* out = reinterpret_cast<float*>(a.out) + (size_t)g * HD + h * kD;
  if (nwaves == 1) {
    out[dg + 4 * jc] = o[0];
    return;
  }
  s_out[wave][dg + 4 * jc] = o[0];
  __syncthreads();
  if (threadIdx.x < kD) {
    float acc = s_out[0][threadIdx.x];
    for (int w = 1; w < nwaves; ++w) acc += s_out[w][threadIdx.x];
    out[threadIdx.x] = acc;
  }
}

// ---- float32 cross-attention -------------------------------------------------
// K is [B, H, E, 64] (head dim contiguous), V is [B, H, 64, E].  Lane = key
// position for the scores (a lane reads its own 256-byte K row), lane = head
// dim for the value product (a lane reads its own row, 64 positions of it).  What
// bounds it at the few rows it is used for is the wait for memory: keys, and values
// where registers allow (WM <= 4 wavefronts), are requested before the queries are
// looked at, and nothing past the length.  us per launch, with one value at a time
// behind the probabilities / with requests for all positions / now:
//   8 items, 6 heads, 64 positions, all valid    8.6 / 5.9 / 5.5
//   64 items, 12 heads, 256, all valid            69 / 22.3 / 20.8
//   64 items, 12 heads, 256, 40 valid            7.7 / 20.2 / 6.2
//   64 items, 12 heads, 512, 60 valid           11.1 / 35.2 / 7.6
//   64 items, 12 heads, 64, 10 valid             4.4 / 6.6 / 4.3
// and with probabilities read from LDS 16 positions at a time, the first wavefront's
// requests in front of the length while workgroups are few, before / now: 8 items, 6
// heads, 64 positions 5.7 / 3.85, 16 x 6 x 256 (100 valid) 7.0 / 5.2, 16 x 6 x 48 5.4 /
// 3.8, 64 x 12 x 64 (10 valid) 4.8 / 4.5, 64 x 12 x 256 (40 valid) 9.0 / 7.6.  What it
// costs: 8 x 6 x 64 with 5 valid 3.7 / 4.2, 128 x 12 x 256, all valid, 36.1 / 37.7.
template <int NQ, int WM>
__global__ void __launch_bounds__(64 * WM)
cross_attn_f32_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) float s_q[NQ][kD];
  __shared__ float s_red[WM][NQ];
  __shared__ __attribute__((aligned(16))) float s_p[NQ][WM * 64];
  __shared__ float s_out[WM][NQ][kD];
  T5D_GATE_READ(a.gate);
  const int h = blockIdx.x, b = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int HD = a.H * kD;
  const float* kbase = reinterpret_cast<const float*>(a.k) +
                       ((size_t)b * a.H + h) * (size_t)a.S * kD;
  const float* vbase = reinterpret_cast<const float*>(a.v) +
                       ((size_t)b * a.H + h) * (size_t)kD * a.S;
  const float* qbase = reinterpret_cast<const float*>(a.q);
  const int j = wave * 64 + lane, jb = wave * 64;
  // keys of this lane's position, values of this lane's row
  float4 key[kD / 4], value[16];
  const auto request_keys = [&](int n) {
    const float4* row =
        reinterpret_cast<const float4*>(kbase + (size_t)min(j, n - 1) * kD);
#pragma unroll
    for (int c = 0; c < kD / 4; ++c) key[c] = row[c];
  };
  constexpr bool kAhead = WM <= 4;
  // (rows of a multiple of 4 floats, aligned: checked by the caller)
  const auto request_values = [&](int n) {
    const float* row = vbase + (size_t)lane * a.S + jb;
    // A whole wavefront's in one go: a lane's 16 loads lie in four lines of 64 bytes, and
    // with addresses formed in between, the loads of 15 other wavefronts come in between
    // and take the lines out of L1 (32 x 12 heads, 900 of 1000 valid, us: before the
    // values were read 16 at a time 40.0, then 43.8, so 36.4).  Up to 4 wavefronts it costs
    // 28 registers, and a third workgroup per CU.
    if (!kAhead && jb + 64 <= n) {
#pragma unroll
      for (int c = 0; c < 16; ++c) value[c] = *reinterpret_cast<const float4*>(row + 4 * c);
      asm volatile("");  // (or the first of them are made one with those below)
      return;
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {  // (what is left out is not looked at)
      if (c % 4 == 0 && jb + 4 * c >= n) break;
      value[c] = *reinterpret_cast<const float4*>(row + min(4 * c, a.S - 4 - jb));
    }
  };
  const bool early = a.early && wave == 0;
  int n = a.index[b];  // (one wait for both)
  if constexpr (kAhead) {
    if (early) {
      request_keys(a.S);
      request_values(a.S);
    }
  }
  T5D_GATE_TEST();
  n = n < 0 ? 0 : (n > a.S ? a.S : n);
  bool uniform = false;
  if (n == 0) { uniform = true; n = a.S; }
  // wavefronts without a position leave (barriers wait for those that are there)
  if (wave * 64 >= n) return;
  const int nwaves = (n + 63) >> 6, threads = 64 * nwaves;
  const int je = min(n, jb + 64);
  // the others': nothing past the length but the last position's keys again and the
  // rest of its sixteen values
  if constexpr (kAhead) {
    if (!early) {
      request_keys(n);
      request_values(n);
    }
  }
  for (int e = threadIdx.x; e < NQ * kD; e += threads) {
    const int qi = e / kD, d = e % kD;
    s_q[qi][d] = qi < a.nq
                     ? qbase[(size_t)(b * a.nq + qi) * a.q_stride + h * kD + d]
                     : 0.f;
  }
  if constexpr (!kAhead) request_keys(n);
  __syncthreads();
  float s[NQ];
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) s[qi] = 0.f;
  if (j < n) {
#pragma unroll
    for (int c = 0; c < kD / 4; ++c) {
      const float4 kv = key[c];
#pragma unroll
      for (int qi = 0; qi < NQ; ++qi) {
        s[qi] = fmaf(s_q[qi][4 * c + 0], kv.x, s[qi]);
        s[qi] = fmaf(s_q[qi][4 * c + 1], kv.y, s[qi]);
        s[qi] = fmaf(s_q[qi][4 * c + 2], kv.z, s[qi]);
        s[qi] = fmaf(s_q[qi][4 * c + 3], kv.w, s[qi]);
      }
    }
  }
  if constexpr (!kAhead) request_values(n);
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) {
    float x = uniform ? 0.f : s[qi];
    x = (j < n) ? x : -INFINITY;
    s[qi] = x;
    const float m = wave_max(x);
    if (lane == 0) s_red[wave][qi] = m;
  }
  __syncthreads();
  float ex[NQ];
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) {
    float m = s_red[0][qi];
    for (int w = 1; w < nwaves; ++w) m = fmaxf(m, s_red[w][qi]);
    ex[qi] = (s[qi] == -INFINITY) ? 0.f : expf(s[qi] - m);
  }
  __syncthreads();
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) {
    const float t = wave_sum(ex[qi]);
    if (lane == 0) s_red[wave][qi] = t;
  }
  __syncthreads();
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) {
    float t = s_red[0][qi];
    for (int w = 1; w < nwaves; ++w) t += s_red[w][qi];
    s_p[qi][j] = ex[qi] / t;
  }
  __syncthreads();
  // value product: lane = head dim, this wavefront's 64 positions
  float o[NQ];
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) o[qi] = 0.f;
  // (a branch per 16 positions: with one per four every probability was a wait for LDS
  // of its own; a masked position's is zero, and its value is not looked at)
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const int jj = jb + 4 * c;
    if (c % 4 == 0 && jj >= je) break;
    const float4 v = make_float4(jj < je ? value[c].x : 0.f, jj + 1 < je ? value[c].y : 0.f,
                                 jj + 2 < je ? value[c].z : 0.f,
                                 jj + 3 < je ? value[c].w : 0.f);
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi) {
      const float4 p = *reinterpret_cast<const float4*>(&s_p[qi][jj]);
      o[qi] = fmaf(p.x, v.x, o[qi]);
      o[qi] = fmaf(p.y, v.y, o[qi]);
      o[qi] = fmaf(p.z, v.z, o[qi]);
      o[qi] = fmaf(p.w, v.w, o[qi]);
    }
  }
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) s_out[wave][qi][lane] = o[qi];
  __syncthreads();
  for (int e = threadIdx.x; e < NQ * kD; e += threads) {
    const int qi = e / kD, d = e % kD;
    if (qi >= a.nq) continue;
    float acc = s_out[0][qi][d];
    for (int w = 1; w < nwaves; ++w) acc += s_out[w][qi][d];
    reinterpret_cast<float*>(a.out)[(size_t)(b * a.nq + qi) * HD + h * kD + d] =
        acc;
  }
}

static void launch_self_f32(AttnArgs a, int rows, hipStream_t s) {
  const int waves = (a.S + 63) / 64;
  dim3 grid(a.H, rows), block(64 * waves);
  a.early = (int64_t)a.H * rows <= 256;
  if (waves <= 4)
    hipLaunchKernelGGL(self_attn_f32_kernel<4>, grid, block, 0, s, a);
  else if (waves <= 8)
    hipLaunchKernelGGL(self_attn_f32_kernel<8>, grid, block, 0, s, a);
  else
    hipLaunchKernelGGL(self_attn_f32_kernel<16>, grid, block, 0, s, a);
}

static void launch_cross_f32(AttnArgs a, int B, hipStream_t s) {
  const int waves = (a.S + 63) / 64;
  a.early = (int64_t)a.H * B <= 256;
  dim3 grid(a.H, B), block(64 * waves);
#define T5D_CROSS_F32(NQ_)                                                        \
  do {                                                                            \
    if (waves <= 4)                                                               \
      hipLaunchKernelGGL((cross_attn_f32_kernel<NQ_, 4>), grid, block, 0, s, a);  \
    else                                                                          \
      hipLaunchKernelGGL((cross_attn_f32_kernel<NQ_, 16>), grid, block, 0, s, a); \
  } while (0)
  if (a.nq == 1) T5D_CROSS_F32(1);
  else if (a.nq == 2) T5D_CROSS_F32(2);
  else if (a.nq <= 4) T5D_CROSS_F32(4);
  else T5D_CROSS_F32(8);
#undef T5D_CROSS_F32
}

int launch_cross_attention_bf16(hipStream_t s, const void* q, const void* k,
                                const void* v, const int32_t* enc_len,
                                void* out, int B, int beams, int H, int E,
                                const void* x, const void* ln, const void* wq,
                                int d, float eps, const int32_t* units);
int launch_self_attention_bf16(hipStream_t s, const void* qkv, void* ck,
                               void* cv, const void* rel_bias,
                               const int32_t* cache_index, void* out, int R,
                               int H, int L, const int32_t* pending,
                               const int32_t* pending_dst, int beams,
                               int value_blocked);

static int check_common(const char* name, int dtype, int H, int S) {
  T5D_REQUIRE(dtype == T5D_F32 || dtype == T5D_BF16, T5D_EINVAL, "%s: dtype %d",
              name, dtype);
  const int el = dtype == T5D_F32 ? 4 : 8;
  T5D_REQUIRE(H > 0 && S > 0 && S % el == 0, T5D_EINVAL,
              "%s: H=%d, length %d must be a positive multiple of %d", name, H,
              S, el);
  T5D_REQUIRE(S <= kMaxWaves * 16 * el, T5D_ELIMIT,
              "%s: length %d beyond the %d positions one workgroup covers",
              name, S, kMaxWaves * 16 * el);
  return T5D_OK;
}

}  // namespace t5d

using namespace t5d;

extern "C" int t5d_self_attention_step(void* stream, int dtype, const void* qkv,
                                       void* cached_key, void* cached_value,
                                       const void* rel_bias,
                                       const int32_t* cache_index, void* out,
                                       int R, int H, int L) {
  int rc = check_common("t5d_self_attention_step", dtype, H, L);
  if (rc) return rc;
  T5D_REQUIRE(qkv && cached_key && cached_value && rel_bias && cache_index &&
                  out && R > 0,
              T5D_EINVAL, "t5d_self_attention_step: null pointer or R=%d", R);
  T5D_REQUIRE(((uintptr_t)cached_key % 16) == 0 &&
                  ((uintptr_t)cached_value % 16) == 0,
              T5D_EINVAL, "t5d_self_attention_step: cache not 16-byte aligned");
  AttnArgs a;
  a.q = qkv; a.k = cached_key; a.v = cached_value; a.rel_bias = rel_bias;
  a.index = cache_index; a.out = out;
  a.H = H; a.S = L; a.nq = 1; a.q_stride = 3 * H * kD;
  a.gate = tls_gate;
  if (dtype == T5D_F32)
    launch_self_f32(a, R, as_stream(stream));
  else
    launch_self_attention_bf16(as_stream(stream), qkv, cached_key, cached_value,
                               rel_bias, cache_index, out, R, H, L, nullptr,
                               nullptr, 1, 0);
  T5D_CHECK_LAUNCH("t5d_self_attention_step");
  return T5D_OK;
}

extern "C" int t5d_self_attention_step_gather(
    void* stream, int dtype, const void* qkv, void* cached_key,
    void* cached_value, const void* rel_bias, const int32_t* cache_index,
    void* out, int B, int beams, int H, int L, const int32_t* pending_src,
    const int32_t* pending_dst, int value_blocked) {
  int rc = check_common("t5d_self_attention_step_gather", dtype, H, L);
  if (rc) return rc;
  T5D_REQUIRE(dtype == T5D_BF16, T5D_EINVAL,
              "t5d_self_attention_step_gather: bfloat16 caches only");
  T5D_REQUIRE(qkv && cached_key && cached_value && rel_bias && cache_index &&
                  out && B > 0 && beams > 0,
              T5D_EINVAL,
              "t5d_self_attention_step_gather: null pointer or B=%d beams=%d", B,
              beams);
  T5D_REQUIRE(pending_src == nullptr ||
                  beams * ((L + 127) / 128) <= kMaxWaves,
              T5D_ELIMIT,
              "t5d_self_attention_step_gather: beams=%d x L=%d needs more than "
              "%d wavefronts per workgroup", beams, L, kMaxWaves);
  T5D_REQUIRE(pending_dst == nullptr || pending_src != nullptr, T5D_EINVAL,
              "t5d_self_attention_step_gather: pending_dst without pending_src");
  T5D_REQUIRE(value_blocked >= 0 && value_blocked <= 3, T5D_EINVAL,
              "t5d_self_attention_step_gather: value_blocked=%d", value_blocked);
  const bool in_place = pending_src != nullptr && pending_dst == nullptr;
  T5D_REQUIRE(value_blocked != 3 || L <= (in_place ? 128 : 256), T5D_ELIMIT,
              "t5d_self_attention_step_gather: the tail layout covers L <= %d "
              "%s (L=%d)", in_place ? 128 : 256,
              in_place ? "for a gather without destination slots" : "", L);
  T5D_REQUIRE(value_blocked != 3 || beams <= 8, T5D_ELIMIT,
              "t5d_self_attention_step_gather: beams=%d (tail layout: 1..8)",
              beams);
  T5D_REQUIRE(!value_blocked || L % 32 == 0, T5D_EINVAL,
              "t5d_self_attention_step_gather: blocked caches need L %% 32 == 0 "
              "(L=%d)", L);
  T5D_REQUIRE(((uintptr_t)cached_key % 16) == 0 &&
                  ((uintptr_t)cached_value % 16) == 0,
              T5D_EINVAL,
              "t5d_self_attention_step_gather: cache not 16-byte aligned");
  launch_self_attention_bf16(as_stream(stream), qkv, cached_key, cached_value,
                             rel_bias, cache_index, out, B * beams, H, L,
                             pending_src, pending_dst, beams, value_blocked);
  T5D_CHECK_LAUNCH("t5d_self_attention_step_gather");
  return T5D_OK;
}

extern "C" int t5d_cross_attention_step(void* stream, int dtype, const void* q,
                                        const void* cross_key,
                                        const void* cross_value,
                                        const int32_t* enc_len, void* out,
                                        int B, int beams, int H, int E,
                                        const int32_t* units) {
  int rc = check_common("t5d_cross_attention_step", dtype, H, E);
  if (rc) return rc;
  T5D_REQUIRE(units == nullptr || dtype == T5D_BF16, T5D_EINVAL,
              "t5d_cross_attention_step: a work order is for bfloat16 only");
  T5D_REQUIRE(q && cross_key && cross_value && enc_len && out && B > 0,
              T5D_EINVAL, "t5d_cross_attention_step: null pointer or B=%d", B);
  T5D_REQUIRE(beams >= 1 && beams <= 8, T5D_ELIMIT,
              "t5d_cross_attention_step: beams=%d (supported: 1..8)", beams);
  T5D_REQUIRE(((uintptr_t)cross_key % 16) == 0 &&
                  ((uintptr_t)cross_value % 16) == 0,
              T5D_EINVAL, "t5d_cross_attention_step: K/V not 16-byte aligned");
  AttnArgs a;
  a.q = q; a.k = const_cast<void*>(cross_key);
  a.v = const_cast<void*>(cross_value); a.rel_bias = nullptr;
  a.index = enc_len; a.out = out;
  a.H = H; a.S = E; a.nq = beams; a.q_stride = H * kD;
  a.gate = tls_gate;
  if (dtype == T5D_F32) {
    T5D_REQUIRE(E <= kMaxWaves * 64, T5D_ELIMIT,
                "t5d_cross_attention_step: float32 covers at most %d positions",
                kMaxWaves * 64);
    launch_cross_f32(a, B, as_stream(stream));
  } else {
    T5D_REQUIRE(E % 32 == 0, T5D_EINVAL,
                "t5d_cross_attention_step: bfloat16 K/V are stored in blocks of "
                "32 positions, E=%d", E);
    launch_cross_attention_bf16(as_stream(stream), q, cross_key, cross_value,
                                enc_len, out, B, beams, H, E, nullptr, nullptr,
                                nullptr, 0, 0.f, units);
  }
  T5D_CHECK_LAUNCH("t5d_cross_attention_step");
  return T5D_OK;
}

// ---- work order of the cross-attention workgroups ---------------------------------
// A cross-attention launch has one workgroup per (item, head) whose work grows
// with the item's valid encoder length.  The dispatcher deals workgroups out
// round-robin (position p goes to XCD p % 8 and, there, to CU (p / 8) % 32), two
// to a CU at most, so with more workgroups than CUs position p shares its CU
// with position p + n_cu, and the launch lasts as long as its most loaded CU.
// This kernel writes the order that evens the CUs out: the heaviest units sit
// alone on a CU, the rest are paired heaviest with lightest; launches of more
// than two rounds get the units by falling length.  One workgroup; B <= 256.
__global__ void __launch_bounds__(256)
cross_units_kernel(const int32_t* __restrict__ enc_len, int B, int H, int E,
                   int n_cu, int32_t* __restrict__ units) {
  __shared__ int s_len[256];
  __shared__ int s_item[256];  // items by falling length (ties: lower index)
  const int tid = threadIdx.x;
  if (tid < B) {
    const int n = enc_len[tid];
    s_len[tid] = n < 0 ? 0 : (n > E ? E : n);
  }
  __syncthreads();
  if (tid < B) {
    const int mine = s_len[tid];
    int rank = 0;
    for (int o = 0; o < B; ++o) {
      const int other = s_len[o];
      rank += (other > mine || (other == mine && o < tid)) ? 1 : 0;
    }
    s_item[rank] = tid;
  }
  __syncthreads();
  const int n = B * H;
  const int pairs = n - n_cu, alone = 2 * n_cu - n;
  for (int r = tid; r < n; r += 256) {
    const int b = s_item[r / H], h = r % H;
    int p = r;
    if (n > n_cu && n <= 2 * n_cu) {
      const int rr = r - alone;
      p = r < alone ? pairs + r : (rr < pairs ? rr : n_cu + (2 * pairs - 1 - rr));
    }
    // an item without a valid key keeps 0: the kernel then attends uniformly
    units[p] = h | (b << 8) | (int)((uint32_t)s_len[b] << 16);
  }
}

extern "C" int t5d_cross_attention_units(void* stream, const int32_t* enc_len,
                                         int B, int H, int E, int32_t* units) {
  T5D_REQUIRE(enc_len && units, T5D_EINVAL,
              "t5d_cross_attention_units: null pointer");
  T5D_REQUIRE(B > 0 && B <= 256 && H > 0 && H <= 256 && E > 0 && E < 32768,
              T5D_ELIMIT,
              "t5d_cross_attention_units: B=%d H=%d (1..256 each), E=%d "
              "(below 32768)", B, H, E);
  static int n_cu = 0;
  if (n_cu == 0) {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) !=
            hipSuccess || v <= 0)
      v = 256;
    n_cu = v;
  }
  hipLaunchKernelGGL(cross_units_kernel, dim3(1), dim3(256), 0,
                     as_stream(stream), enc_len, B, H, E, n_cu, units);
  T5D_CHECK_LAUNCH("t5d_cross_attention_units");
  return T5D_OK;
}

extern "C" int t5d_cross_attention_step_norm_q(
    void* stream, int dtype, int w_dtype, const void* x, const void* ln_scale,
    float eps, const void* query_kernel, const void* cross_key,
    const void* cross_value, const int32_t* enc_len, void* out, int B,
    int beams, int H, int E, int d, const int32_t* units) {
  int rc = check_common("t5d_cross_attention_step_norm_q", dtype, H, E);
  if (rc) return rc;
  T5D_REQUIRE(dtype == T5D_BF16 && w_dtype == T5D_BF16, T5D_EINVAL,
              "t5d_cross_attention_step_norm_q: bfloat16 activations and "
              "weights only");
  T5D_REQUIRE(x && ln_scale && query_kernel && cross_key && cross_value &&
                  enc_len && out && B > 0,
              T5D_EINVAL,
              "t5d_cross_attention_step_norm_q: null pointer or B=%d", B);
  T5D_REQUIRE(beams >= 1 && beams <= 8, T5D_ELIMIT,
              "t5d_cross_attention_step_norm_q: beams=%d (supported: 1..8)",
              beams);
  T5D_REQUIRE(E <= 512 && E % 32 == 0 && d >= 64 && d % 64 == 0 && d <= 1024,
              T5D_ELIMIT,
              "t5d_cross_attention_step_norm_q: E=%d (multiple of 32, <= 512), "
              "d=%d (multiple of 64, <= 1024)", E, d);
  T5D_REQUIRE(((uintptr_t)cross_key % 16) == 0 &&
                  ((uintptr_t)cross_value % 16) == 0 &&
                  ((uintptr_t)x % 16) == 0 && ((uintptr_t)ln_scale % 16) == 0 &&
                  ((uintptr_t)query_kernel % 16) == 0,
              T5D_EINVAL,
              "t5d_cross_attention_step_norm_q: operands not 16-byte aligned");
  launch_cross_attention_bf16(as_stream(stream), nullptr, cross_key, cross_value,
                              enc_len, out, B, beams, H, E, x, ln_scale,
                              query_kernel, d, eps, units);
  T5D_CHECK_LAUNCH("t5d_cross_attention_step_norm_q");
  return T5D_OK;
}
