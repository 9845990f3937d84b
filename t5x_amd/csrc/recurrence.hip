// Linear recurrences over a matrix state per head, with one decay per key
// channel, for sequences that are fed in portions of any length:
//
//   S <- diag(g_t) S;  u = v_t  or, with the delta rule,  u = beta_t (v_t - S^T k_t);
//   S <- S + k_t u^T;  o_t = S^T q_t
//
// S [D, Dv] is float32 and lives in a slot per sequence; a portion that starts at
// position 0 starts from zeros whatever the slot holds.  Around it, in float32:
// an optional short causal convolution with silu on q, k and v (its last inputs
// live in the slot too, a ring by position), optional unit norms of q and k, the
// decay from a low-rank projection, and the norm and gate of the read-out.
//
// Short portions run as prepare (a wavefront per token and head vector), a scan
// token by token, and finish.  Long ones are cut into chunks of 16 tokens.  With
// P_t the product of the decays of a chunk up to token t, the state S0 before it
// and X the solution of (I + diag(beta) A) X = diag(beta) R, A[t][s] = sum_d k_t
// (P_t / P_s) k_s for s < t, and B the same with q_t for s <= t,
//   Wk = X(k P), Us = X(v):       u = Us - Wk S0          (no delta rule: u = v)
//   Qs = q P - B Wk, Os = B Us:   o = Os + Qs S0
//   S  = diag(P_16) S0 + Kh^T u,  Kh_t = k_t P_16 / P_t
// Everything but the products with S0 and the state is independent of the other
// chunks: one kernel forms it for all chunks at once, from the projections on
// (quotients of decays as running products, which are at most 1), a second walks
// the chunks with three matrix products each, in float32 on the matrix cores.
// A step of one token per sequence is one kernel per (sequence, head) that reads
// and writes the state once.
#include <algorithm>

#include "common.h"
#include "gemm_tiles.h"

namespace t5d {

struct RecArgs {
  t5d_recurrence a;
  t5d_ragged b;
  // float32 scratch of a portion
  float *wq, *wk, *wv, *wbeta, *wo;
  float* wchunk;  // chunked portions: the chunks' operands (ChunkLayout)
  int chunks;     // of the longest portion: the chunk kernel's grid
  int32_t* order;  // chunked portions, or null: [S] the sequences, longest first
  int C;  // channels of the convolution
  const int32_t* gate;
};

__device__ __forceinline__ float exp_f(float z) {
  return __builtin_amdgcn_exp2f(z * 1.4426950408889634f);
}
__device__ __forceinline__ float sigmoid_f(float z) {
  return 1.0f / (1.0f + exp_f(-z));
}
__device__ __forceinline__ float softplus_f(float z) {
  return z > 20.f ? z : log1pf(expf(z));
}

// Logarithm of the decay of a key channel of head h from its biased projection z.
__device__ __forceinline__ float log_decay_of(const t5d_recurrence& a, float z, int h) {
  if (a.decay == T5D_DECAY_SIGMOID_POWER) return -softplus_f(-z) * a.decay_power;
  return -expf(a.A_log[h]) * softplus_f(z);
}

// The same of channel c from its projection.
__device__ __forceinline__ float log_decay(const t5d_recurrence& a, float z, int h,
                                           int c) {
  return log_decay_of(a, z + a.decay_bias[(size_t)h * a.D + c], h);
}

// The same for the chunk kernel, which spent most of its instructions on them:
// quotients as a reciprocal and one step of Newton (within an ulp, as the division),
// log2(1 + e^z) with what rounding took from 1 + e added back to first order.  Error of
// float32 outputs against float64 (96 tokens, 24 inputs each), with the library's functions,
// divisions and a substitution per column / with these and the inverse below:
//   delta rule, heads of 64, 4 taps    slow decays 1.53e-7 / 1.50e-7, fast 1.33e-7 / 1.22e-7
//   delta rule, heads of 128, no taps              2.17e-7 / 2.14e-7       1.49e-7 / 1.38e-7
//   no delta rule, heads of 128                    2.11e-7 / 2.12e-7       1.42e-7 / 1.40e-7
//   no delta rule, heads of 64, 4 taps             1.10e-7 / 1.10e-7       1.17e-7 / 1.17e-7
//   delta rule, one key for all tokens 7.45e-7 / 7.50e-7, keys 1 % apart 9.88e-7 / 1.02e-6
__device__ __forceinline__ float reciprocal_f(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return x > 1e30f ? r : fmaf(fmaf(-x, r, 1.0f), r, r);  // (infinity: 0)
}
__device__ __forceinline__ float sigmoid_quick(float z) {
  return reciprocal_f(1.0f + exp_f(-z));
}
__device__ __forceinline__ float softplus_log2(float z) {
  constexpr float kLog2e = 1.4426950408889634f;
  const float e = __builtin_amdgcn_exp2f(-kLog2e * fabsf(z));
  const float u = 1.0f + e;
  const float lost = (e - (u - 1.0f)) * kLog2e;
  const float l = fmaf(lost, __builtin_amdgcn_rcpf(u), __builtin_amdgcn_logf(u));
  return fmaf(fmaxf(z, 0.0f), kLog2e, l);
}

// One channel of q, k or v of the token at row m: the projection itself, or its
// causal convolution and silu.  `first`: row of the portion's first token; cc:
// channel of the convolution; x: value at row m.
template <typename T>
__device__ __forceinline__ float conv_channel(const RecArgs& g, int m, int first,
                                              int pos, int slot, int col, int cc,
                                              float x) {
  const t5d_recurrence& a = g.a;
  const float* w = a.conv + (size_t)cc * a.taps;
  float s = x * w[a.taps - 1];
  const T* ring = reinterpret_cast<const T*>(a.conv_ring) +
                  (size_t)slot * a.taps * g.C + cc;
  for (int j = 1; j < a.taps; ++j) {
    if (pos - j < 0) break;
    const float v = m - j >= first
                        ? to_f32<T>(reinterpret_cast<const T*>(
                              a.proj)[(size_t)(m - j) * a.ld_proj + col])
                        : to_f32<T>(ring[(size_t)((pos - j) % a.taps) * g.C]);
    s = fmaf(v, w[a.taps - 1 - j], s);
  }
  return s * sigmoid_f(s);
}

// ---- prepare ----------------------------------------------------------------------
// Vectors of a token: (with a convolution or unit norms) G queries, G keys, H
// values; then H decays.
template <typename T>
__global__ void __launch_bounds__(256)
recurrence_prepare_kernel(RecArgs g) {
  T5D_GATED(g.gate);
  const t5d_recurrence& a = g.a;
  const int lane = threadIdx.x & 63;
  const bool qkv = a.taps > 0 || a.unit;
  const int nq = qkv ? 2 * a.G + a.H : 0, nvec = nq + a.H;
  const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= (int64_t)g.b.M * nvec) return;
  const int m = unit / nvec, vec = unit % nvec;
  const T* p = reinterpret_cast<const T*>(a.proj) + (size_t)m * a.ld_proj;
  if (vec >= nq) {
    const int h = vec - nq;
    float* z = a.low + (size_t)m * a.ld_low + a.off_z + (size_t)h * a.D;
    for (int c = lane; c < a.D; c += 64) z[c] = log_decay(a, z[c], h, c);
    if (a.delta && lane == 0)
      g.wbeta[(size_t)m * a.H + h] = sigmoid_f(to_f32<T>(p[a.off_beta + h]));
    return;
  }
  const bool query = vec < a.G, key = !query && vec < 2 * a.G;
  const int h = query ? vec : key ? vec - a.G : vec - 2 * a.G;
  const int n = query || key ? a.D : a.Dv;
  const int col0 = query ? a.off_q + h * a.D : key ? a.off_k + h * a.D
                                                   : a.off_v + h * a.Dv;
  const int cc0 = query ? h * a.D : key ? (a.G + h) * a.D : 2 * a.G * a.D + h * a.Dv;
  float* out = query ? g.wq + ((size_t)m * a.G + h) * a.D
               : key ? g.wk + ((size_t)m * a.G + h) * a.D
                     : g.wv + ((size_t)m * a.H + h) * a.Dv;
  const int seq = g.b.tok_seq[m], pos = g.b.tok_pos[m];
  const int first = g.b.seq_off[seq], slot = g.b.seq_slot[seq];
  float ss = 0.f;
  for (int c = lane; c < n; c += 64) {
    float x = to_f32<T>(p[col0 + c]);
    if (a.taps > 0)
      x = conv_channel<T>(g, m, first, pos, slot, col0 + c, cc0 + c, x);
    ss = fmaf(x, x, ss);
    out[c] = x;
  }
  if (!(query || key)) return;
  float f = query ? a.q_scale : 1.f;
  if (a.unit) f /= sqrtf(wave_sum(ss) + a.unit_eps);
  for (int c = lane; c < n; c += 64) out[c] *= f;  // this lane's own stores
}

// ---- scan ---------------------------------------------------------------------------
// A workgroup owns 16 columns of a head's state, a wavefront 4 of them: lane
// (kl, column) holds the rows d = 64 e + 4 kl + j of its column.  Columns never
// interact.  Keys, queries and decays of 8 tokens at a time go through LDS, the
// next 8 are on their way meanwhile.
template <int E4, bool DELTA, typename TQ>
__global__ void __launch_bounds__(256)
recurrence_scan_kernel(RecArgs g, const TQ* q_rows, const TQ* k_rows,
                       const TQ* v_rows, int ldq, int ldk, int ldv, float q_scale) {
  constexpr int DP = 64 * E4, TS = 8, NP = TS * DP / 256;
  __shared__ __align__(16) float s_k[TS][DP];
  __shared__ __align__(16) float s_q[TS][DP];
  __shared__ __align__(16) float s_g[TS][DP];
  __shared__ float s_v[TS][16];
  __shared__ float s_b[TS];
  T5D_GATED(g.gate);
  const t5d_recurrence& a = g.a;
  const int h = blockIdx.y, seq = blockIdx.z, hg = h / (a.H / a.G);
  const int off = g.b.seq_off[seq], T = g.b.seq_off[seq + 1] - off;
  const int start = g.b.seq_start[seq], slot = g.b.seq_slot[seq];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kl = lane & 15, cw = wave * 4 + (lane >> 4);
  const int col = blockIdx.x * 16 + cw;
  const bool col_ok = col < a.Dv;
  if (T <= 0) return;

  float* state = a.state + ((size_t)slot * a.H + h) * a.D * a.Dv + col;
  float st[E4 * 4];
#pragma unroll
  for (int e = 0; e < E4 * 4; ++e) {
    const int d = 64 * (e >> 2) + 4 * kl + (e & 3);
    st[e] = start > 0 && col_ok && d < a.D ? state[(size_t)d * a.Dv] : 0.f;
  }
  const TQ* q = q_rows + (size_t)off * ldq + (size_t)hg * a.D;
  const TQ* k = k_rows + (size_t)off * ldk + (size_t)hg * a.D;
  const TQ* v = v_rows + (size_t)off * ldv + (size_t)h * a.Dv;
  const float* lg = a.low + (size_t)off * a.ld_low + a.off_z + (size_t)h * a.D;
  float* o = g.wo + ((size_t)off * a.H + h) * a.Dv + col;

  float pk[NP], pq[NP], pg[NP], pv = 0.f, pb = 0.f;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = threadIdx.x + 256 * i, t = t0 + e / DP, d = e % DP;
      const bool ok = t < T && d < a.D;
      pk[i] = ok ? to_f32<TQ>(k[(size_t)t * ldk + d]) : 0.f;
      pq[i] = ok ? to_f32<TQ>(q[(size_t)t * ldq + d]) * q_scale : 0.f;
      pg[i] = ok ? lg[(size_t)t * a.ld_low + d] : 0.f;
    }
    if (threadIdx.x < TS * 16) {
      const int t = t0 + threadIdx.x / 16, c = blockIdx.x * 16 + threadIdx.x % 16;
      pv = t < T && c < a.Dv ? to_f32<TQ>(v[(size_t)t * ldv + (threadIdx.x % 16) +
                                            blockIdx.x * 16])
                             : 0.f;
    } else if (DELTA && threadIdx.x < TS * 16 + TS) {
      const int t = t0 + threadIdx.x - TS * 16;
      pb = t < T ? g.wbeta[(size_t)(off + t) * a.H + h] : 0.f;
    }
  };
  fetch(0);
  for (int t0 = 0; t0 < T; t0 += TS) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = threadIdx.x + 256 * i;
      s_k[e / DP][e % DP] = pk[i];
      s_q[e / DP][e % DP] = pq[i];
      s_g[e / DP][e % DP] = expf(pg[i]);
    }
    if (threadIdx.x < TS * 16) s_v[threadIdx.x / 16][threadIdx.x % 16] = pv;
    else if (DELTA && threadIdx.x < TS * 16 + TS) s_b[threadIdx.x - TS * 16] = pb;
    __syncthreads();
    if (t0 + TS < T) fetch(t0 + TS);
    const int n = min(TS, T - t0);
    for (int t = 0; t < n; ++t) {
      float kk[E4 * 4], qq[E4 * 4];
      float s0 = 0.f, s1 = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int e = 0; e < E4; ++e) {
        const float4 x = *reinterpret_cast<const float4*>(&s_k[t][64 * e + 4 * kl]);
        const float4 y = *reinterpret_cast<const float4*>(&s_q[t][64 * e + 4 * kl]);
        const float4 w = *reinterpret_cast<const float4*>(&s_g[t][64 * e + 4 * kl]);
        kk[4 * e] = x.x; kk[4 * e + 1] = x.y; kk[4 * e + 2] = x.z; kk[4 * e + 3] = x.w;
        qq[4 * e] = y.x; qq[4 * e + 1] = y.y; qq[4 * e + 2] = y.z; qq[4 * e + 3] = y.w;
        st[4 * e] *= w.x; st[4 * e + 1] *= w.y;
        st[4 * e + 2] *= w.z; st[4 * e + 3] *= w.w;
        if (DELTA) {
          s0 = fmaf(st[4 * e], x.x, s0);
          s1 = fmaf(st[4 * e + 1], x.y, s1);
          s0 = fmaf(st[4 * e + 2], x.z, s0);
          s1 = fmaf(st[4 * e + 3], x.w, s1);
        }
      }
      float u = s_v[t][cw];
      if (DELTA) u = s_b[t] * (u - lanes16_sum(s0 + s1));
#pragma unroll
      for (int e = 0; e < E4 * 4; e += 2) {
        st[e] = fmaf(kk[e], u, st[e]);
        st[e + 1] = fmaf(kk[e + 1], u, st[e + 1]);
        o0 = fmaf(st[e], qq[e], o0);
        o1 = fmaf(st[e + 1], qq[e + 1], o1);
      }
      const float r = lanes16_sum(o0 + o1);
      if (kl == 0 && col_ok) o[(size_t)(t0 + t) * a.H * a.Dv] = r;
    }
  }
#pragma unroll
  for (int e = 0; e < E4 * 4; ++e) {
    const int d = 64 * (e >> 2) + 4 * kl + (e & 3);
    if (col_ok && d < a.D) state[(size_t)d * a.Dv] = st[e];
  }
}

// ---- chunks ---------------------------------------------------------------------------
constexpr int kChunk = 16;

// A sequence's first chunk in the scratch memory: the sequences before it have
// at most this many chunks together.
__host__ __device__ __forceinline__ size_t chunk_base(int64_t first_token, int seq) {
  return (size_t)(first_token / kChunk + seq);
}

// What the chunk kernel leaves per (chunk, head), in floats, in the
// operand order of v_mfma_f32_16x16x4_f32: lane (x, g) of 16 x 4 holds element
// (row x, k g) of the left operand, (k g, column x) of the right one, and rows
// 4 g + i of column x of the result.  Step i of a product takes k = 4 g + i from
// lane (x, g), so that a result tile is the right operand of the next product as
// it stands; a left operand is then one float4 per lane and tile:
//   wk, qs [tile of 16 channels][lane]: channels 16 tile + 4 g + i of token x
//   kh     [tile][lane]: tokens 4 g + i, channel 16 tile + x
//   us, os [tile of 16 columns][lane]: tokens 4 g + i, column 16 tile + x
//   pc     [channel]: the chunk's whole decay
struct ChunkLayout {
  int dp, vp;
  __host__ __device__ ChunkLayout(int dp_, int vp_) : dp(dp_), vp(vp_) {}
  __host__ __device__ size_t wk() const { return 0; }
  __host__ __device__ size_t qs() const { return (size_t)kChunk * dp; }
  __host__ __device__ size_t kh() const { return (size_t)2 * kChunk * dp; }
  __host__ __device__ size_t us() const { return (size_t)3 * kChunk * dp; }
  __host__ __device__ size_t os() const { return us() + (size_t)kChunk * vp; }
  __host__ __device__ size_t pc() const { return os() + (size_t)kChunk * vp; }
  __host__ __device__ size_t size() const { return pc() + dp; }
};

// The chunk's columns of q, k, the decay and v, one per thread and 512 per round, into
// LDS: q, k and v through the convolution and silu if there is one (TM: at least its
// taps).  Two columns of a thread are requested before either is used, and rows past
// the end are the last one again (no branches between the loads); such tokens have no
// key, no query, no value and no decay.  chunk, n: which chunk, its tokens.
template <int TM, int DP, typename T>
__device__ __forceinline__ void chunk_columns(const RecArgs& g, int chunk, int n, int m0,
                                              int h, int seq, float* s_q, float* s_k,
                                              float* s_g, float* s_v, int vp, int vs) {
  constexpr int C = kChunk, LS = DP + 4, N = TM > 0 ? TM : 1;
  const t5d_recurrence& a = g.a;
  const int tid = threadIdx.x, hg = h / (a.H / a.G);
  const int slot = g.b.seq_slot[seq], pos0 = g.b.seq_start[seq] + chunk * C;
  const bool power = a.decay == T5D_DECAY_SIGMOID_POWER;
  const float rate = power ? a.decay_power : expf(a.A_log[h]);
  struct Column {
    int kind, c;        // 0 q, 1 k, 2 decay, 3 v; column within it
    float x[C];
    float w[N], before[N];  // before[j]: the value j tokens before the chunk
  };
  const auto load = [&](Column& y, int u) {
    y.kind = min(__builtin_amdgcn_readfirstlane(u) / DP, 3);  // (DP % 64 == 0)
    y.c = u - y.kind * DP;
    const int c = y.c < (y.kind == 3 ? a.Dv : a.D) ? y.c : 0;
    if (y.kind == 2) {
      const float* z = a.low + (size_t)m0 * a.ld_low + a.off_z + (size_t)h * a.D + c;
#pragma unroll
      for (int t = 0; t < C; ++t) y.x[t] = z[(size_t)min(t, n - 1) * a.ld_low];
      y.w[0] = a.decay_bias[(size_t)h * a.D + c];
      return;
    }
    const int col = (y.kind == 0 ? a.off_q + hg * a.D
                     : y.kind == 1 ? a.off_k + hg * a.D : a.off_v + h * a.Dv) + c;
    const int cc = (y.kind == 0 ? hg * a.D
                    : y.kind == 1 ? (a.G + hg) * a.D : 2 * a.G * a.D + h * a.Dv) + c;
    const T* p = reinterpret_cast<const T*>(a.proj) + (size_t)m0 * a.ld_proj + col;
#pragma unroll
    for (int t = 0; t < C; ++t) y.x[t] = to_f32<T>(p[(size_t)min(t, n - 1) * a.ld_proj]);
    if constexpr (TM > 0) {
      const T* ring = reinterpret_cast<const T*>(a.conv_ring) +
                      (size_t)slot * a.taps * g.C + cc;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        y.w[j] = j < a.taps ? a.conv[(size_t)cc * a.taps + a.taps - 1 - j] : 0.f;
        y.before[j] = 0.f;
        if (j > 0 && j < a.taps) {
          if (chunk * C >= j)
            y.before[j] = to_f32<T>(p[-(ptrdiff_t)j * a.ld_proj]);
          else if (pos0 >= j)
            y.before[j] = to_f32<T>(ring[(size_t)((pos0 - j) % a.taps) * g.C]);
        }
      }
    }
  };
  const auto finish = [&](const Column& y) {
    float v[C];
    if (y.kind == 2) {
      const float sign = power ? -1.f : 1.f;
#pragma unroll
      for (int t = 0; t < C; ++t) {  // the exponential of log_decay
        const float z = sign * (y.x[t] + y.w[0]);
        v[t] = __builtin_amdgcn_exp2f(-rate * softplus_log2(z));
      }
    } else if constexpr (TM > 0) {
#pragma unroll
      for (int t = 0; t < C; ++t) {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < N; ++j)
          sum = fmaf(y.w[j], t >= j ? y.x[t >= j ? t - j : 0] : y.before[t >= j ? 0 : j - t],
                     sum);
        v[t] = sum * sigmoid_quick(sum);
      }
    } else {
#pragma unroll
      for (int t = 0; t < C; ++t) v[t] = y.x[t];
    }
    if (y.c >= (y.kind == 3 ? vp : DP)) return;
    const bool there = y.c < (y.kind == 3 ? a.Dv : a.D);
    float* dst = (y.kind == 0 ? s_q : y.kind == 1 ? s_k : y.kind == 2 ? s_g : s_v) + y.c;
    const int stride = y.kind == 3 ? vs : LS;
    const float none = y.kind == 2 ? 1.f : 0.f;
#pragma unroll
    for (int t = 0; t < C; ++t) dst[t * stride] = there && t < n ? v[t] : none;
  };
  for (int u = tid; u < 3 * DP + vp; u += 512) {
    Column y0, y1;
    const bool more = __builtin_amdgcn_readfirstlane(u) + 256 < 3 * DP + vp;
    load(y0, u);
    if (more) load(y1, u + 256);
    finish(y0);
    if (more) finish(y1);
  }
}

constexpr int kChunkTaps = 8;  // longest convolution of the chunk kernel

// Columns of q, k, v and the decay through convolution, silu and norms; A and B on
// the vector ALUs, k_s decayed on its way down the chunk; then, with the delta rule,
// T = (I + diag(beta) A)^-1 diag(beta), 16 x 16, and everything that is applied to
// whole columns on the matrix cores: Wk = T (k P), Us = T v, and with M = B T
// Qs = q P - M (k P), Os = M v.
// What bounds it: vector instructions (59 % of their slots by the counters; 1714 per
// wavefront, half of them silu and decays) with four workgroups per CU, then 42 KB written
// per chunk and head.  4 x 4096 tokens, 8 heads of 128: delta rule 160 us, gated linear attention
// 103 us; 301 and 240 us with the triangular solve and the products with B down each
// column on the vector ALUs, divisions instead of sigmoid_quick, the library's
// logarithm, and loads that branches kept from being in flight together.
template <int DP, bool DELTA, typename T>
__global__ void __launch_bounds__(256, DP <= 128 ? 4 : DP <= 256 ? 2 : 1)
recurrence_chunk_kernel(RecArgs g) {
  constexpr int LS = DP + 4, C = kChunk;
  __shared__ __align__(16) float s_k[C * LS];
  __shared__ __align__(16) float s_q[C * LS];
  __shared__ __align__(16) float s_g[C * LS];
  __shared__ __align__(16) float s_a[C][C];
  __shared__ __align__(16) float s_b[C][C];
  __shared__ __align__(16) float s_t[C][C];
  __shared__ float s_beta[C];
  extern __shared__ float s_v[];  // [C][vp + 4]
  T5D_GATED(g.gate);
  const t5d_recurrence& a = g.a;
  const int chunk = blockIdx.x, h = blockIdx.y, seq = blockIdx.z;
  const int off = g.b.seq_off[seq], len = g.b.seq_off[seq + 1] - off;
  const int tid = threadIdx.x;
  if (g.order && chunk == 0 && h == 0) {
    // where the sequence stands by its length, for the chain kernel
    __shared__ int s_longer;
    if (tid == 0) s_longer = 0;
    __syncthreads();
    int longer = 0;
    for (int i = tid; i < g.b.S; i += 256) {
      const int other = g.b.seq_off[i + 1] - g.b.seq_off[i];
      longer += other > len || (other == len && i < seq);
    }
    atomicAdd(&s_longer, longer);
    __syncthreads();
    if (tid == 0) g.order[s_longer] = seq;
  }
  const int n = min(C, len - chunk * C);
  if (n <= 0) return;
  const int m0 = off + chunk * C;
  const int vp = (a.Dv + 15) / 16 * 16, vs = vp + 4;
  if (a.taps == 0)
    chunk_columns<0, DP, T>(g, chunk, n, m0, h, seq, s_q, s_k, s_g, s_v, vp, vs);
  else if (a.taps <= 4)
    chunk_columns<4, DP, T>(g, chunk, n, m0, h, seq, s_q, s_k, s_g, s_v, vp, vs);
  else
    chunk_columns<kChunkTaps, DP, T>(g, chunk, n, m0, h, seq, s_q, s_k, s_g, s_v, vp, vs);
  if (DELTA && tid < C)
    s_beta[tid] = tid < n ? sigmoid_f(to_f32<T>(reinterpret_cast<const T*>(
                                a.proj)[(size_t)(m0 + tid) * a.ld_proj + a.off_beta + h]))
                          : 0.f;
  s_a[tid >> 4][tid & 15] = 0.f;
  s_b[tid >> 4][tid & 15] = 0.f;
  __syncthreads();
  {
    // unit norms and the query's factor: 8 lanes per row of q, then of k
    const bool query = tid < 128;
    float* row = (query ? s_q : s_k) + ((tid >> 3) & 15) * LS + 4 * (tid & 7);
    float f = query ? a.q_scale : 1.f;
    if (a.unit) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < DP / 32; ++e) {
        const float4 x = *reinterpret_cast<const float4*>(row + 32 * e);
        ss = fmaf(x.x, x.x, ss); ss = fmaf(x.y, x.y, ss);
        ss = fmaf(x.z, x.z, ss); ss = fmaf(x.w, x.w, ss);
      }
      ss += dpp_move<kDppXor1>(ss);
      ss += dpp_move<kDppXor2>(ss);
      ss += dpp_move<kDppHalfMirror>(ss);
      f /= sqrtf(ss + a.unit_eps);
    }
    if (a.unit || query) {
#pragma unroll
      for (int e = 0; e < DP / 32; ++e) {
        float4 x = *reinterpret_cast<const float4*>(row + 32 * e);
        x.x *= f; x.y *= f; x.z *= f; x.w *= f;
        *reinterpret_cast<float4*>(row + 32 * e) = x;
      }
    }
  }
  __syncthreads();
  {
    // B and, with the delta rule, A: half of the wavefronts each, 16 lanes (without
    // it 32) per source token, which walk t = s .. 15 with k_s decayed on the way;
    // source j, then source 15 - j: 17 steps for everyone.
    constexpr int LPS = DELTA ? 16 : 32, E = (DP + 4 * LPS - 1) / (4 * LPS);
    const bool keys = DELTA && tid >= 128;
    const int j = (tid / LPS) & 7, c0 = 4 * (tid % LPS);
    const float* other = keys ? s_k : s_q;
    float(*dst)[C] = keys ? s_a : s_b;
    float4 x[E];
#pragma unroll
    for (int i = 0; i <= C; ++i) {
      const bool second = i >= C - j;
      const int s = second ? C - 1 - j : j, t = second ? i - 1 : j + i;
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int c = c0 + 4 * LPS * e;
        if (DP % (4 * LPS) != 0 && c >= DP) continue;
        const int o = t * LS + c;
        if (t == s) {
          x[e] = *reinterpret_cast<const float4*>(s_k + o);
        } else {
          const float4 w = *reinterpret_cast<const float4*>(s_g + o);
          x[e].x *= w.x; x[e].y *= w.y; x[e].z *= w.z; x[e].w *= w.w;
        }
        const float4 y = *reinterpret_cast<const float4*>(other + o);
        sum = fmaf(x[e].x, y.x, sum); sum = fmaf(x[e].y, y.y, sum);
        sum = fmaf(x[e].z, y.z, sum); sum = fmaf(x[e].w, y.w, sum);
      }
      sum = lanes16_sum(sum);
      if constexpr (LPS == 32) {
        const auto w = __builtin_amdgcn_permlane16_swap(
            __float_as_uint(sum), __float_as_uint(sum), false, false);
        sum = __uint_as_float(w[0]) + __uint_as_float(w[1]);
      }
      if (tid % LPS == 0 && (!keys || t > s)) dst[t][s] = sum;
    }
  }
  __syncthreads();

  const ChunkLayout lay(DP, vp);
  float* w = g.wchunk + ((chunk_base(off, seq) + chunk) * a.H + h) * lay.size();
  if (tid >= 128) {
    // a column of T per thread
    if (DELTA && tid < 128 + C) {
      const int c = tid - 128;
      float x[C];
#pragma unroll
      for (int t = 0; t < C; ++t) {
        float r = t == c ? 1.f : 0.f;
#pragma unroll
        for (int s = 0; s < t; ++s) r = fmaf(-s_a[t][s], x[s], r);
        x[t] = r * s_beta[t];
        s_t[t][c] = x[t];
      }
    }
  } else {
    // a channel per thread: k P, q P, Kh and the whole decay
    for (int c = tid; c < DP; c += 128) {
      float k[C], run = 1.f, back = 1.f;
#pragma unroll
      for (int t = 0; t < C; ++t) {
        const int o = t * LS + c;
        run *= s_g[o];
        k[t] = s_k[o];
        s_k[o] = k[t] * run;
        s_q[o] *= run;
      }
      w[lay.pc() + c] = run;
#pragma unroll
      for (int t = C - 1; t >= 0; --t) {
        const float gt = s_g[t * LS + c];
        s_g[t * LS + c] = k[t] * back;
        back *= gt;
      }
    }
  }
  __syncthreads();
  // Tiles of 16 channels, then of 16 value columns, dealt to the wavefronts.
  const int lane = tid & 63, x = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const auto four = [](const float* p, float (&v)[4]) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
  };
  const auto times = [](const float (&l)[4], const float (&r)[4], f32x4_v acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(l[i], r[i], acc, 0, 0, 0);
    return acc;
  };
  const auto put = [](float* p, int at, f32x4_v v) {
    reinterpret_cast<float4*>(p)[at] = make_float4(v[0], v[1], v[2], v[3]);
  };
  const f32x4_v zero = (f32x4_v){0.f, 0.f, 0.f, 0.f};
  // The products multiply the zeros above the diagonals of T and M by what later
  // tokens hold, which is no zero where that is infinite or NaN: an operand with such
  // a value goes down its column over s <= t alone, so that a token never reaches an
  // earlier one, as on the token by token path.
  const auto not_finite = [](const float (&v)[4]) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) bad |= !(fabsf(v[i]) < INFINITY);
    return __builtin_amdgcn_ballot_w64(bad) != 0;
  };
  const auto down = [](const float (&row)[C], int t, const float* p, int stride) {
    float sum = 0.f;
#pragma unroll 1
    for (int s = 0; s <= t; ++s) sum = fmaf(row[s], p[s * stride], sum);
    return sum;
  };
  float tm[4], bm[4], mm[4];  // rows x of T, B and M, columns 4 g + i
  four(&s_b[x][4 * g4], bm);
#pragma unroll
  for (int i = 0; i < 4; ++i) mm[i] = bm[i];
  if (DELTA) {
    four(&s_t[x][4 * g4], tm);
    float tc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) tc[i] = s_t[4 * g4 + i][x];
    if (not_finite(tc)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mm[i] = 0.f;
#pragma unroll 1
        for (int k = 4 * g4 + i; k <= x; ++k)
          mm[i] = fmaf(s_b[x][k], s_t[k][4 * g4 + i], mm[i]);
      }
    } else {
      const f32x4_v m = times(tc, bm, zero);  // M^T: rows 4 g + i, column x
#pragma unroll
      for (int i = 0; i < 4; ++i) mm[i] = m[i];
    }
    // M for `down` (A is no longer needed; every wavefront writes the same)
    *reinterpret_cast<float4*>(&s_a[x][4 * g4]) =
        make_float4(mm[0], mm[1], mm[2], mm[3]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  const float(*s_m)[C] = DELTA ? s_a : s_b;
  for (int tile = wave; tile < DP / 16; tile += 4) {
    const int at = tile * 64 + lane;
    f32x4_v q;
    {
      const float4 f = *reinterpret_cast<const float4*>(s_q + x * LS + 16 * tile + 4 * g4);
      q = (f32x4_v){f.x, f.y, f.z, f.w};
    }
    const int o = 4 * g4 * LS + 16 * tile + x;
    if (DELTA) {
      float r[4], minus[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[i] = s_k[o + i * LS];
        minus[i] = -r[i];
      }
      if (not_finite(r)) {
        f32x4_v k;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* column = s_k + 16 * tile + 4 * g4 + i;
          k[i] = down(s_t[x], x, column, LS);
          q[i] -= down(s_m[x], x, column, LS);
        }
        put(w + lay.wk(), at, k);
      } else {
        put(w + lay.wk(), at, times(r, tm, zero));
        q = times(minus, mm, q);
      }
    }
    put(w + lay.qs(), at, q);
    put(w + lay.kh(), at,
        (f32x4_v){s_g[o], s_g[o + LS], s_g[o + 2 * LS], s_g[o + 3 * LS]});
  }
  for (int tile = wave; tile < vp / 16; tile += 4) {
    const int at = tile * 64 + lane;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = s_v[(4 * g4 + i) * vs + 16 * tile + x];
    f32x4_v u = (f32x4_v){v[0], v[1], v[2], v[3]}, y;
    if (not_finite(v)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* column = s_v + 16 * tile + x;
        if (DELTA) u[i] = down(s_t[4 * g4 + i], 4 * g4 + i, column, vs);
        y[i] = down(s_m[4 * g4 + i], 4 * g4 + i, column, vs);
      }
    } else if (DELTA) {
      u = times(tm, v, zero);
      y = times(mm, v, zero);
    } else {
      // tokens in their order: the last ones weigh most where decays are fast
      float b[4], late[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        b[i] = s_b[x][4 * i + g4];
        late[i] = s_v[(4 * i + g4) * vs + 16 * tile + x];
      }
      y = times(b, late, zero);
    }
    put(w + lay.us(), at, u);
    put(w + lay.os(), at, y);
  }
}

// Walks the chunks of one (sequence, head) for 16 NC value columns.  Each of 4
// wavefronts holds NTW tiles of 16 channels x 16 columns of the state per NC.
// What bounds it where sequences are few: the chain of a step at one wavefront per SIMD (24
// dependent matrix products = 770 of its 2000 cycles, the exchange of partial sums behind
// one barrier, the requests).  Nothing that the state does not need stands in front of the
// barrier; a read-out's parts wait for the next step's.  Where they are many: matrix
// instructions and the operands' way into a CU, 24 KB per step that columns side by side
// share, so two column tiles (NC = 2) go together once one alone has more than two
// workgroups per CU (the line in launch_chunks); and how evenly the sequences fall on the
// CUs, so the longest start first (RecArgs::order).  Chunk, chain and finish kernel together,
// us, 8 heads of 128, delta rule / without, with the read-out in front of the barrier, one
// column tile and sequences as they stand -> now:
//   4 x 2048 tokens            213 -> 204    136 -> 132
//   1 x 4096                   248 -> 244    163 -> 157
//   40 of 3 to 611             281 -> 238    198 -> 162
//   16 x 300                   120 -> 112     81 -> 76.5  (16 x 300 of 4 heads, one tile:
//                               72 -> 72      50 -> 49.5)
template <int NTW, bool DELTA, int NC>
__global__ void __launch_bounds__(256, NTW <= 2 ? 2 : 1)
recurrence_chain_kernel(RecArgs g) {
  constexpr int DP = 64 * NTW;
  __shared__ float4 s_u[2][NC][4][64];
  __shared__ float4 s_o[2][NC][4][64];
  T5D_GATED(g.gate);
  const t5d_recurrence& a = g.a;
  // The workgroups of one (sequence, head) read the same operands: consecutive
  // block ids go round-robin over the 8 XCDs, so theirs are 8 apart.
  const int vp = (a.Dv + 15) / 16 * 16, vts = (vp / 16 + NC - 1) / NC;
  const int pair = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / vts);
  if (pair >= a.H * g.b.S) return;
  const int vt = NC * ((blockIdx.x >> 3) % vts), h = pair % a.H;
  const int seq = g.order ? g.order[pair / a.H] : pair / a.H;
  const int off = g.b.seq_off[seq], len = g.b.seq_off[seq + 1] - off;
  if (len <= 0) return;
  const int start = g.b.seq_start[seq], slot = g.b.seq_slot[seq];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = lane & 15, g4 = lane >> 4;
  const int col = 16 * vt + x;  // and 16 further on
  const ChunkLayout lay(DP, vp);
  const int nc = (len + kChunk - 1) / kChunk;

  float* state = a.state + ((size_t)slot * a.H + h) * a.D * a.Dv + col;
  f32x4_v st[NC][NTW];
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * (wave * NTW + t) + 4 * g4 + i;
        st[n][t][i] = start > 0 && col + 16 * n < a.Dv && d < a.D
                          ? state[(size_t)d * a.Dv + 16 * n] : 0.f;
      }
  const size_t row = (size_t)a.H * a.Dv;  // of the read-outs
  float* out = g.wo + (size_t)off * row + (size_t)h * a.Dv + col +
               (size_t)(4 * g4 + wave) * row;

  struct Operands {
    float4 wk[NTW], qs[NTW], kh[NTW], pc[NTW], us[NC];
    float os[NC];
  };
  // Operands: a uniform base per chunk, which stops at the last one, and offsets
  // within a chunk that never change.  (A column tile past the end has none: it takes the
  // first one's, for columns that are not stored.)
  const size_t stride = (size_t)a.H * lay.size() * sizeof(float);
  char* next = reinterpret_cast<char*>(
      g.wchunk + (chunk_base(off, seq) * a.H + h) * lay.size());
  int to_load = nc;  // chunks not yet requested
  const uint32_t at = (wave * NTW * 64 + lane) * 16;
  const uint32_t at_pc = (wave * NTW * 4 + g4) * 16;
  const uint32_t at_us = (vt * 64 + lane) * 16, at_os = at_us + 4 * wave;
  const uint32_t further = vt + 1 < vp / 16 ? 1024 : 0;
  auto load = [&](Operands& o) {
#if defined(__HIP_DEVICE_COMPILE__)  // (buffer descriptors are no host type)
    // (the base moves with scalar additions)
    const __amdgpu_buffer_rsrc_t chunk =
        __builtin_amdgcn_make_buffer_rsrc(next, 0, 0x7fffffff, 0x00020000);
    const auto piece = [&](size_t of, uint32_t o) {
      return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                            chunk, (int)o, (int)(4 * of), 0));
    };
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      if (DELTA) o.wk[t] = piece(lay.wk(), at + 1024 * t);
      o.qs[t] = piece(lay.qs(), at + 1024 * t);
      o.kh[t] = piece(lay.kh(), at + 1024 * t);
      o.pc[t] = piece(lay.pc(), at_pc + 64 * t);
    }
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      o.us[n] = piece(lay.us(), at_us + n * further);
      // (only the row this wavefront stores is used)
      o.os[n] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(
                     chunk, (int)(at_os + n * further), (int)(4 * lay.os()), 0));
    }
    next += --to_load > 0 ? stride : 0;
#endif
  };
  // The read-out of a chunk, tokens 4 g + wave: its product's parts meet behind the barrier
  // of the step after it.
  float os[NC], y[NC][4];
  const auto fetch_out = [&](int c) {
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int p = 0; p < 4; ++p)
        y[n][p] = reinterpret_cast<const float*>(&s_o[c & 1][n][p][lane])[wave];
  };
  const auto read_out = [&](int c) {
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const float sum = (((os[n] + y[n][0]) + y[n][1]) + y[n][2]) + y[n][3];
      if (kChunk * c + 4 * g4 + wave < len && col + 16 * n < a.Dv) out[16 * n] = sum;
    }
    out += kChunk * row;
  };
  // A step: u's product and the exchange of the wavefronts' parts; behind the barrier,
  // while they are on their way, the requests for a later chunk and the read-out's
  // product; then the state's update.
  auto step = [&](const Operands& o, Operands& later, int c) {
    const int buf = c & 1;
    if (DELTA) {
      f32x4_v u[NC];
#pragma unroll
      for (int n = 0; n < NC; ++n) u[n] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        const float wk[4] = {o.wk[t].x, o.wk[t].y, o.wk[t].z, o.wk[t].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int n = 0; n < NC; ++n)
            u[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wk[i], st[n][t][i], u[n], 0, 0, 0);
      }
#pragma unroll
      for (int n = 0; n < NC; ++n)
        s_u[buf][n][wave][lane] = make_float4(u[n][0], u[n][1], u[n][2], u[n][3]);
      __builtin_amdgcn_sched_barrier(0);
    }
    f32x4_v old[NC][NTW];
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        old[n][t] = st[n][t];
        st[n][t][0] *= o.pc[t].x; st[n][t][1] *= o.pc[t].y;
        st[n][t][2] *= o.pc[t].z; st[n][t][3] *= o.pc[t].w;
      }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    float4 p[NC][4];
    if (DELTA) {
#pragma unroll
      for (int n = 0; n < NC; ++n)
#pragma unroll
        for (int w = 0; w < 4; ++w) p[n][w] = s_u[buf][n][w][lane];
    }
    fetch_out(c + 1);  // (the chunk before; of the first nothing is stored)
    __builtin_amdgcn_sched_barrier(0);
    load(later);
    f32x4_v r[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) r[n] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      const float qs[4] = {o.qs[t].x, o.qs[t].y, o.qs[t].z, o.qs[t].w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NC; ++n)
          r[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(qs[i], old[n][t][i], r[n], 0, 0, 0);
    }
    float uu[NC][4];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      uu[n][0] = o.us[n].x; uu[n][1] = o.us[n].y;
      uu[n][2] = o.us[n].z; uu[n][3] = o.us[n].w;
      if (DELTA) {
        uu[n][0] -= (p[n][0].x + p[n][1].x) + (p[n][2].x + p[n][3].x);
        uu[n][1] -= (p[n][0].y + p[n][1].y) + (p[n][2].y + p[n][3].y);
        uu[n][2] -= (p[n][0].z + p[n][1].z) + (p[n][2].z + p[n][3].z);
        uu[n][3] -= (p[n][0].w + p[n][1].w) + (p[n][2].w + p[n][3].w);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        const float kh[4] = {o.kh[t].x, o.kh[t].y, o.kh[t].z, o.kh[t].w};
#pragma unroll
        for (int n = 0; n < NC; ++n)
          st[n][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kh[i], uu[n][i], st[n][t], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NC; ++n)
      s_o[buf][n][wave][lane] = make_float4(r[n][0], r[n][1], r[n][2], r[n][3]);
    if (c > 0) read_out(c - 1);
#pragma unroll
    for (int n = 0; n < NC; ++n) os[n] = o.os[n];
  };
  // The operands of the next chunks are on their way while one is multiplied.  The
  // compiler waits for all of them at the head of a loop, hence 16 steps per round, 12 with
  // two column tiles (three sets of operands: a round ends on the set it began with).
  constexpr int DEPTH = NTW > 4 ? 2 : NC > 1 ? 3 : 4;
  constexpr int ROUND = NTW <= 2 ? NC > 1 ? 12 : 16 : DEPTH;
  static_assert(ROUND % DEPTH == 0, "operands of one chunk, steps of another");
  Operands o[DEPTH];
#pragma unroll
  for (int i = 0; i + 1 < DEPTH; ++i) load(o[i]);
  for (int c0 = 0; c0 < nc; c0 += ROUND) {
#pragma unroll
    for (int i = 0; i < ROUND; ++i) {
      if (c0 + i >= nc) break;
      step(o[i % DEPTH], o[(i + DEPTH - 1) % DEPTH], c0 + i);
    }
  }
  __syncthreads();
  fetch_out(nc - 1);
  read_out(nc - 1);
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * (wave * NTW + t) + 4 * g4 + i;
        if (col + 16 * n < a.Dv && d < a.D) state[(size_t)d * a.Dv + 16 * n] = st[n][t][i];
      }
}

// The convolution's last inputs of a portion, written once nothing of the portion
// reads the ring any more.
template <typename T>
__global__ void __launch_bounds__(256)
recurrence_conv_tail_kernel(RecArgs g) {
  T5D_GATED(g.gate);
  const t5d_recurrence& a = g.a;
  const int seq = blockIdx.y;
  const int off = g.b.seq_off[seq], len = g.b.seq_off[seq + 1] - off;
  const int cc = blockIdx.x * 256 + threadIdx.x;
  if (cc >= g.C) return;
  const int qk = a.G * a.D;
  const int col = cc < qk ? a.off_q + cc
                  : cc < 2 * qk ? a.off_k + cc - qk : a.off_v + cc - 2 * qk;
  T* ring = reinterpret_cast<T*>(a.conv_ring) +
            (size_t)g.b.seq_slot[seq] * a.taps * g.C + cc;
  for (int t = max(0, len - (a.taps - 1)); t < len; ++t)
    ring[(size_t)((g.b.seq_start[seq] + t) % a.taps) * g.C] =
        reinterpret_cast<const T*>(a.proj)[(size_t)(off + t) * a.ld_proj + col];
}

// ---- read-out: norm, gate -----------------------------------------------------------
__device__ __forceinline__ float out_gate_of(const t5d_recurrence& a, float z) {
  return a.gate == T5D_GATE_SIGMOID_LOW ? sigmoid_f(z) : z * sigmoid_f(z);
}
template <typename T>
__device__ __forceinline__ float out_gate(const t5d_recurrence& a, int m, int h,
                                          int c) {
  if (a.gate == T5D_GATE_SIGMOID_LOW)
    return out_gate_of(a, a.low[(size_t)m * a.ld_low + a.off_low_gate +
                                (size_t)h * a.Dv + c]);
  return out_gate_of(a, to_f32<T>(reinterpret_cast<const T*>(
      a.proj)[(size_t)m * a.ld_proj + a.off_gate + (size_t)h * a.Dv + c]));
}

// A wavefront per (token, head); with VEC 4 columns per lane, two heads of up to
// 128 columns per wavefront.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256)
recurrence_finish_kernel(RecArgs g) {
  T5D_GATED(g.gate);
  const t5d_recurrence& a = g.a;
  const int lane = threadIdx.x & 63;
  if constexpr (VEC) {
    const int64_t unit = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
    const bool on = unit < (int64_t)g.b.M * a.H;
    const int m = on ? unit / a.H : 0, h = on ? unit % a.H : 0;
    const int c = 4 * (lane & 31);
    const bool ok = on && c < a.Dv;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f), z = o;
    if (ok) {
      o = *reinterpret_cast<const float4*>(g.wo + (size_t)unit * a.Dv + c);
      if (a.gate == T5D_GATE_SIGMOID_LOW) {
        z = *reinterpret_cast<const float4*>(a.low + (size_t)m * a.ld_low +
                                             a.off_low_gate + (size_t)h * a.Dv + c);
      } else {
        const T* p = reinterpret_cast<const T*>(a.proj) + (size_t)m * a.ld_proj +
                     a.off_gate + (size_t)h * a.Dv + c;
        z = make_float4(to_f32<T>(p[0]), to_f32<T>(p[1]), to_f32<T>(p[2]),
                        to_f32<T>(p[3]));
      }
    }
    float ss = lanes16_sum(o.x * o.x + o.y * o.y + o.z * o.z + o.w * o.w);
    const auto w = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(ss), __float_as_uint(ss), false, false);
    ss = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    if (!ok) return;
    const float inv = 1.0f / sqrtf(ss / (float)a.Dv + a.eps);
    const bool silu = a.gate != T5D_GATE_SIGMOID_LOW;
    auto put = [&](float v, float zz, float nw) {
      return v * inv * nw * (silu ? zz * sigmoid_f(zz) : sigmoid_f(zz));
    };
    const float y0 = put(o.x, z.x, a.norm[c]), y1 = put(o.y, z.y, a.norm[c + 1]);
    const float y2 = put(o.z, z.z, a.norm[c + 2]), y3 = put(o.w, z.w, a.norm[c + 3]);
    T* out = reinterpret_cast<T*>(a.out) + (size_t)m * a.ld_out + (size_t)h * a.Dv + c;
    if constexpr (sizeof(T) == 2) {
      *reinterpret_cast<uint2*>(out) =
          make_uint2(pack_bf16x2(y0, y1), pack_bf16x2(y2, y3));
    } else {
      *reinterpret_cast<float4*>(out) = make_float4(y0, y1, y2, y3);
    }
    return;
  }
  const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= (int64_t)g.b.M * a.H) return;
  const int m = unit / a.H, h = unit % a.H;
  const float* o = g.wo + (size_t)unit * a.Dv;
  float ss = 0.f;
  for (int c = lane; c < a.Dv; c += 64) ss = fmaf(o[c], o[c], ss);
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)a.Dv + a.eps);
  T* out = reinterpret_cast<T*>(a.out) + (size_t)m * a.ld_out + (size_t)h * a.Dv;
  for (int c = lane; c < a.Dv; c += 64)
    Act<T>::store(out + c, o[c] * inv * a.norm[c] * out_gate<T>(a, m, h, c));
}

// ---- one token per sequence ------------------------------------------------------------
// One workgroup per (sequence, head), a wavefront per 32 columns and at least four, as
// the first four form q, k, v and the decay, one each: lane (quad, dg) holds rows
// dg + 8 i of 4 neighbouring columns, so a load instruction reads 8 runs of 128 bytes.
// The kernel is one chain of waits, so everything is requested at its start, in the
// order in which it is needed (loads are waited for in order): the projections, the
// taps and the ring of the convolution, the output's gate, then the state; q, k, v and
// the decay are formed while the state is on its way.  Without the delta rule, where
// there is little to form, the state comes first: it then keeps the memory busy from
// the start in launches of two workgroups per CU and more (8 heads of 128, 128 tokens:
// 23.1 -> 21.0 us; 64 tokens: 10.4 -> 10.8).
// us per launch, with loads in the convolution's own loop, behind the state, and the
// gate's at the end / now (rows of the state past the last are not requested, by the
// group of 8 x R; one token, then 64, 128, 256):
//   delta rule, 8 heads of 128 x 128, 4 taps   7.2 14.4 29.1 51.7 /  5.9 11.7 23.9 43.8
//   delta rule, 8 heads of 64 x 64, 4 taps     6.0  8.0  9.4 15.5 /  4.3  6.0  8.4 15.6
//   delta rule, 4 heads of 200 x 200, 4 taps  11.8 22.3 43.5 81.2 / 11.1 21.8 41.9 79.4
//   delta rule, 4 heads of 256 x 256, 4 taps  12.1 28.9 55.5  123 / 11.2 27.9 52.9  107
//   delta rule, 4 heads of 32 x 32, 2 taps     6.3  6.6  6.7  7.3 /  3.9  4.2  4.6  6.0
//   no delta rule, 8 heads of 128 x 128        5.8 11.4 21.7 42.6 /  5.0 10.8 21.0 40.6
//   no delta rule, 4 heads of 48 x 64          4.3  4.8  5.6  6.7 /  3.7  4.2  4.9  6.7
// (64 states of 8 x 128 x 128 take 13.7 us at the rate of a large copy from memory.)
// EXACT: heads as wide as the template (32, 64 or 128 channels of keys and of values) and
// taps that are all requested ahead; nothing is tested then: with 128, 2100 instructions
// do instead of 3480, which a lone launch has to fetch (8 heads, one token, in a model's
// step: delta rule 8.0 -> 6.2 us, without 7.3 -> 5.6; launches behind one another, 1 / 64
// rows of 8 heads: 6.1 / 11.7 -> 5.0 / 10.3, of 64 x 64 4.6 / 6.2 -> 3.9 / 5.5, of 32 x 32
// 4.1 / 4.8 -> 3.5 / 4.2).  Heads of 256 have two taps ahead and no registers to gain.
// LOWP > 0: the low-rank stage too, of LOWP pairs of k-tiles.  Every wavefront multiplies the
// token's inputs by its part of the head's columns (one row, in all 16 of the matrix cores;
// summed as t5d_dense does, so with its bits), and the decays are formed where their z lies.
template <int DI, bool DELTA, typename T, bool EXACT, int LOWP>
__global__ void __launch_bounds__(512)
recurrence_step_kernel(RecArgs g) {
  constexpr int DP = 8 * DI;
  constexpr bool LOW = LOWP > 0;
  constexpr int TPW = DP >= 64 ? DP / 64 : 1;  // LOW: column tiles of 16 per wavefront
  static_assert(!LOW || (EXACT && sizeof(T) == 2), "which heads have the low-rank stage");
  __shared__ float s_lg[LOW ? DP : 1];
  __shared__ float s_q[DP], s_k[DP], s_g[DP];
  __shared__ __align__(16) float s_v[256];
  __shared__ __align__(16) float s_o[256];
  __shared__ float s_b;
  T5D_GATE_READ(g.gate);
  const t5d_recurrence& a = g.a;
  const int h = blockIdx.x % a.H, m = blockIdx.x / a.H, hg = h / (a.H / a.G);
  const int pos = g.b.seq_start[m], slot = g.b.seq_slot[m];
  const int D = EXACT ? DP : a.D, Dv = EXACT ? DP : a.Dv;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int quad = lane & 7, dg = lane >> 3;
  const int col = 4 * (8 * wave + quad);
  const bool col_ok = EXACT || col < Dv;
  const T* p = reinterpret_cast<const T*>(a.proj) + (size_t)m * a.ld_proj;
  // role 0, 1, 2: channels lane + 64 u of q, k, v; role 3: of the decay (the first four
  // wavefronts, there whatever the columns, take one each)
  constexpr int U = EXACT ? (DP + 63) / 64 : 4;  // groups of 64 channels
  constexpr int NT = DI <= 16 ? 4 : 2;  // taps requested ahead (registers)
  const int ring0 = a.taps > 0 ? pos % a.taps : 0;
  // (kept as loaded: a conversion here would wait for the load)
  T now[U], past[U][NT - 1];
  float tap[U][NT];
  const auto channels = [&](int role) { return role == 2 ? Dv : D; };
  const auto column = [&](int role) {
    return role == 0 ? a.off_q + hg * D
           : role == 1 ? a.off_k + hg * D : a.off_v + h * Dv;
  };
  const auto channel = [&](int role) {
    return role == 0 ? hg * D
           : role == 1 ? (a.G + hg) * D : 2 * a.G * D + h * Dv;
  };
  const T* ring = reinterpret_cast<const T*>(a.conv_ring) +
                  (size_t)slot * a.taps * g.C;
  // (tiles of z, then of the gate; a wavefront past the head's columns has none)
  const bool low_gate = a.gate == T5D_GATE_SIGMOID_LOW;
  const bool has_low = LOW && 16 * TPW * wave < DP;
  uint4 low_in[LOW ? 2 * LOWP : 1], low_w[LOW ? 2 : 1][TPW][LOW ? 2 * LOWP : 1];
  float low_bias = 0.f;
  const int low_c = min(16 * TPW * wave + (lane & (16 * TPW - 1)), DP - 1);
  const auto request_low = [&] {
    if constexpr (LOW) {
      const uint4* in = reinterpret_cast<const uint4*>(p + a.off_low) + (lane >> 4);
#pragma unroll
      for (int k = 0; k < 2 * LOWP; ++k) low_in[k] = in[4 * k];
      low_bias = a.decay_bias[(size_t)h * DP + low_c];
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        if (which == 1 && !low_gate) break;
        const int tile = ((which ? a.off_low_gate : a.off_z) + h * DP) / 16 + TPW * wave;
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
          for (int k = 0; k < 2 * LOWP; ++k)
            low_w[which][t][k] = reinterpret_cast<const uint4*>(
                a.low_w)[((size_t)(tile + t) * 2 * LOWP + k) * 64 + lane];
      }
    }
  };
  const auto form_low = [&] {
    if constexpr (LOW) {
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        if (which == 1 && !low_gate) break;
        float z[TPW];
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
          f32x4_v acc[LOWP];
#pragma unroll
          for (int q = 0; q < LOWP; ++q) {
            acc[q] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 2 * q; k < 2 * q + 2; ++k) {
              Frag x, w;
              x.u = low_in[k];
              w.u = low_w[which][t][k];
              acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, w.v, acc[q], 0, 0, 0);
            }
          }
          z[t] = LOWP > 1 ? acc[0][0] + acc[LOWP - 1][0] : acc[0][0];
        }
        // (every group of 16 lanes holds all tiles: lane l takes its l / 16th)
        float v = z[0];
        if constexpr (TPW > 1) v = (lane & 16) ? z[1] : z[0];
        if (lane < 16 * TPW) {
          if (which == 0) s_g[low_c] = expf(log_decay_of(a, v + low_bias, h));
          else s_lg[low_c] = v;
        }
      }
    }
  };
  const auto request = [&](int role) {
    if (LOW && role == 3) return;
    if (role == 3) {
#pragma unroll
      for (int u = 0; u < (DP + 63) / 64; ++u) {
        const int c = min(lane + 64 * u, D - 1);
        tap[u][0] = a.decay_bias[(size_t)h * D + c];
        tap[u][1] = a.low[(size_t)m * a.ld_low + a.off_z + (size_t)h * D + c];
      }
      return;
    }
    const int n = channels(role);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!EXACT && 64 * u >= n) break;
      const int c = min(lane + 64 * u, n - 1), cc = channel(role) + c;
      now[u] = p[column(role) + c];
      if (a.taps == 0) continue;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        // (taps and places beyond the sequence's start: read, not used)
        tap[u][j] = a.conv[(size_t)cc * a.taps + max(a.taps - 1 - j, 0)];
        const int at = ring0 - j < 0 ? max(ring0 - j + a.taps, 0) : ring0 - j;
        if (j > 0) past[u][j - 1] = ring[(size_t)at * g.C + cc];
      }
    }
  };
  float* state = a.state + ((size_t)slot * a.H + h) * D * Dv + col;
  float4 st[DI];
  const auto request_state = [&] {
    if constexpr (EXACT) {  // (a sequence's first token: not looked at)
      if (DP < 128 && 32 * wave >= DP) return;  // (there for its role alone)
#pragma unroll
      for (int i = 0; i < DI; ++i)
        st[i] = *reinterpret_cast<const float4*>(state + (size_t)(dg + 8 * i) * Dv);
    } else if (pos > 0 && col_ok) {
      constexpr int R = DELTA && DI == 32 ? 1 : 4;  // rows of 8 per test of the size
#pragma unroll
      for (int i = 0; i < DI; i += R) {
        const bool there = i == 0 || 8 * i < D;
#pragma unroll
        for (int e = i; e < i + R; ++e) {
          st[e] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (there)  // (past the last row the last one again)
            st[e] = *reinterpret_cast<const float4*>(
                state + (size_t)min(dg + 8 * e, D - 1) * Dv);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < DI; ++i) st[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  if (!DELTA) request_state();
  if (wave < 4) request(wave);
  if (has_low) request_low();
  const T beta_z = p[DELTA ? a.off_beta + h : 0];
  // the output channel of this lane
  const int co = 64 * wave + lane;
  const int cg = EXACT ? co % Dv : min(co, Dv - 1);
  const float norm = a.norm[cg];
  // (each from a place that is there; one of them is used)
  const float gate_low =
      LOW ? 0.f
          : a.low[(size_t)m * a.ld_low + (low_gate ? a.off_low_gate + h * Dv + cg : a.off_z)];
  const T gate_z = (low_gate ? p : p + a.off_gate + (size_t)h * Dv)[low_gate ? 0 : cg];
  if (DELTA) request_state();
  T5D_GATE_TEST();
  const auto form = [&](int role) {
    if (role == 3) {
#pragma unroll
      for (int u = 0; !LOW && u < (DP + 63) / 64; ++u) {
        const int c = lane + 64 * u;
        if (c < DP)
          s_g[c] = c < D ? expf(log_decay_of(a, tap[u][1] + tap[u][0], h)) : 0.f;
      }
      if (DELTA && lane == 0) s_b = sigmoid_f(to_f32<T>(beta_z));
      return;
    }
    const int n = channels(role), pad = role == 2 ? n : DP;
    float x[U];
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = lane + 64 * u;
      x[u] = 0.f;
      if (c < n) {
        x[u] = to_f32<T>(now[u]);
        if (a.taps > 0) {
          const int cc = channel(role) + c;
          float v = x[u] * tap[u][0];
#pragma unroll
          for (int j = 1; j < NT; ++j)
            if (j < a.taps && pos - j >= 0)
              v = fmaf(to_f32<T>(past[u][j - 1]), tap[u][j], v);
          for (int j = NT; !EXACT && j < a.taps && pos - j >= 0; ++j)
            v = fmaf(to_f32<T>(ring[(size_t)((pos - j) % a.taps) * g.C + cc]),
                     a.conv[(size_t)cc * a.taps + a.taps - 1 - j], v);
          x[u] = v * sigmoid_f(v);
          reinterpret_cast<T*>(a.conv_ring)[((size_t)slot * a.taps + ring0) * g.C +
                                            cc] = now[u];
        }
        ss = fmaf(x[u], x[u], ss);
      }
    }
    float f = role == 0 ? a.q_scale : 1.f;
    if (a.unit && role < 2) f /= sqrtf(wave_sum(ss) + a.unit_eps);
    float* dst = role == 0 ? s_q : role == 1 ? s_k : s_v;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (lane + 64 * u < pad) dst[lane + 64 * u] = x[u] * f;
  };
  if (wave < 4) form(wave);
  if (has_low) form_low();
  __syncthreads();
  // (a wavefront that was there for its role; barriers wait for those that stay)
  if (32 * wave >= Dv) return;
  if (EXACT && pos <= 0) {
#pragma unroll
    for (int i = 0; i < DI; ++i) st[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (D < DP) {  // rows past the last were read from it
#pragma unroll
    for (int i = 0; i < DI; ++i)
      if (dg + 8 * i >= D) st[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < DI; ++i) {
    const float w = s_g[dg + 8 * i];
    st[i].x *= w; st[i].y *= w; st[i].z *= w; st[i].w *= w;
    if (DELTA) {
      const float k = s_k[dg + 8 * i];
      r.x = fmaf(st[i].x, k, r.x); r.y = fmaf(st[i].y, k, r.y);
      r.z = fmaf(st[i].z, k, r.z); r.w = fmaf(st[i].w, k, r.w);
    }
  }
  // sum over the 8 row groups: lanes ^8, ^16, ^32
  auto over_rows = [](float v) { return rows_sum(v + lane_xor8(v)); };
  float4 u = col_ok ? *reinterpret_cast<const float4*>(s_v + col)
                    : make_float4(0.f, 0.f, 0.f, 0.f);
  if (DELTA) {
    const float beta = s_b;
    u.x = beta * (u.x - over_rows(r.x)); u.y = beta * (u.y - over_rows(r.y));
    u.z = beta * (u.z - over_rows(r.z)); u.w = beta * (u.w - over_rows(r.w));
  }
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < DI; ++i) {
    const float k = s_k[dg + 8 * i], q = s_q[dg + 8 * i];
    st[i].x = fmaf(k, u.x, st[i].x); st[i].y = fmaf(k, u.y, st[i].y);
    st[i].z = fmaf(k, u.z, st[i].z); st[i].w = fmaf(k, u.w, st[i].w);
    o.x = fmaf(st[i].x, q, o.x); o.y = fmaf(st[i].y, q, o.y);
    o.z = fmaf(st[i].z, q, o.z); o.w = fmaf(st[i].w, q, o.w);
    const int d = dg + 8 * i;
    if (EXACT || (col_ok && d < D))
      *reinterpret_cast<float4*>(state + (size_t)d * Dv) = st[i];
  }
  o.x = over_rows(o.x); o.y = over_rows(o.y);
  o.z = over_rows(o.z); o.w = over_rows(o.w);
  if (dg == 0 && col_ok) *reinterpret_cast<float4*>(s_o + col) = o;
  __syncthreads();
  if (co - lane >= Dv) return;
  float ss = 0.f;
  for (int c = lane; c < Dv; c += 64) ss = fmaf(s_o[c], s_o[c], ss);
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)Dv + a.eps);
  if (co < Dv)
    Act<T>::store(reinterpret_cast<T*>(a.out) + (size_t)m * a.ld_out +
                      (size_t)h * Dv + co,
                  s_o[co] * inv * norm *
                      out_gate_of(a, !low_gate ? to_f32<T>(gate_z)
                                     : LOW     ? s_lg[cg]
                                               : gate_low));
}

// Whether a step forms its low-rank columns itself: where heads are as wide as the kernel's
// variant, up to the rows measured.  Steps of 8 layers (6 of them recurrences, heads of 128,
// 64 to 128 inputs), us with a dense layer in front / so, rows 1, 8, 64, 256: 8 heads (width
// 1024) 224.7 / 216.2, 302 / 287, 438 / 424, 1114 / 1090, rows 512 1589 / 1551; 16 heads
// 357 / 341, 468 / 451, 785 / 773, 2013 / 1971.  Launches behind one another, us, dense layer
// and step / so, 64 inputs, rows 1, 64, 128, 256, delta rule: 32 heads of 32 6.0 / 4.5, 10.6 /
// 9.0, 15.7 / 14.2; 16 of 64 6.4 / 4.6, 10.4 / 8.7, 16.1 / 15.1, 28.5 / 24.8; 8 of 128 7.5 /
// 5.9, 13.8 / 11.4, 25.8 / 24.1, 47.6 / 43.9; without it 5.4 / 3.7, 8.9 / 6.8, 13.0 / 10.5; 5.7
// / 3.6, 9.1 / 7.5, 13.5 / 12.0, 26.5 / 22.7; 6.8 / 4.6, 12.8 / 10.1, 25.1 / 22.4, 45.9 / 41.7.
// With 128 inputs up to 1 us of it goes: 32 heads of 32 with 128 rows 15.8 / 15.5, 16 of 64 16.3 /
// 16.8, 256 rows 28.7 / 27.2, 8 of 128 48.1 / 44.9.  (Of 512 rows alone 91.4 / 98.3, in the
// steps above it is the faster one.)
static bool low_rides(const t5d_recurrence& a, int64_t rows) {
  return a.dtype == T5D_BF16 && a.D == a.Dv && (a.D == 32 || a.D == 64 || a.D == 128) &&
         a.taps <= 4 && (a.low_k == 64 || a.low_k == 128) && a.off_z % 16 == 0 &&
         (a.gate != T5D_GATE_SIGMOID_LOW || a.off_low_gate % 16 == 0) &&
         a.off_low % 8 == 0 && a.ld_proj % 8 == 0 &&
         // (what t5d_dense refuses is left for it to refuse)
         a.low_n % 16 == 0 && a.ld_low >= a.low_n &&
         ((uintptr_t)a.proj | (uintptr_t)a.low_w | (uintptr_t)a.low) % 16 == 0 &&
         rows * a.H <= 4096;
}

template <bool DELTA, typename T>
static void launch_step(hipStream_t s, const RecArgs& g) {
  const dim3 grid(g.b.S * g.a.H), block(64 * std::max(4, (g.a.Dv + 31) / 32));
#define T5D_RSL(DI_, EXACT_, LOWP_)                                                     \
  hipLaunchKernelGGL((recurrence_step_kernel<DI_, DELTA, T, EXACT_, LOWP_>), grid, block, \
                     0, s, g)
#define T5D_RS(DI_, EXACT_) T5D_RSL(DI_, EXACT_, 0)
  const bool exact = g.a.D == g.a.Dv && g.a.taps <= 4;
  if constexpr (sizeof(T) == 2) {
    if (g.a.low_w != nullptr) {  // (low_rides)
#define T5D_RSW(DI_)                             \
  do {                                           \
    if (g.a.low_k == 64) T5D_RSL(DI_, true, 1);  \
    else T5D_RSL(DI_, true, 2);                  \
  } while (0)
      if (g.a.D == 32) T5D_RSW(4);
      else if (g.a.D == 64) T5D_RSW(8);
      else T5D_RSW(16);
#undef T5D_RSW
      return;
    }
  }
  if (exact && g.a.D == 32) T5D_RS(4, true);
  else if (g.a.D <= 32) T5D_RS(4, false);
  else if (exact && g.a.D == 64) T5D_RS(8, true);
  else if (g.a.D <= 64) T5D_RS(8, false);
  else if (exact && g.a.D == 128) T5D_RS(16, true);
  else if (g.a.D <= 128) T5D_RS(16, false);
  else T5D_RS(32, false);
#undef T5D_RS
#undef T5D_RSL
}

template <bool DELTA, typename TQ>
static void launch_scan(hipStream_t s, const RecArgs& g, const TQ* q, const TQ* k,
                        const TQ* v, int ldq, int ldk, int ldv, float q_scale) {
  const dim3 grid((g.a.Dv + 15) / 16, g.a.H, g.b.S), block(256);
#define T5D_SC(E_)                                                               \
  hipLaunchKernelGGL((recurrence_scan_kernel<E_, DELTA, TQ>), grid, block, 0, s, \
                     g, q, k, v, ldq, ldk, ldv, q_scale)
  if (g.a.D <= 64) T5D_SC(1);
  else if (g.a.D <= 128) T5D_SC(2);
  else if (g.a.D <= 256) T5D_SC(4);
  else T5D_SC(8);
#undef T5D_SC
}

template <bool DELTA, typename T>
static void launch_chunks(hipStream_t s, const RecArgs& g) {
  const int vts = (g.a.Dv + 15) / 16, pairs = g.a.H * g.b.S;
  const dim3 grid(g.chunks, g.a.H, g.b.S), block(256);
  const dim3 chain((pairs + 7) / 8 * 8 * vts);
  const size_t lds = (size_t)kChunk * (vts * 16 + 4) * sizeof(float);
  const bool two = (int64_t)pairs * vts > 512;  // (see recurrence_chain_kernel)
#define T5D_CH(E_)                                                               \
  do {                                                                           \
    hipLaunchKernelGGL((recurrence_chunk_kernel<64 * E_, DELTA, T>), grid, block, \
                       lds, s, g);                                               \
    if (E_ <= 2 && two)                                                          \
      hipLaunchKernelGGL((recurrence_chain_kernel<E_, DELTA, E_ <= 2 ? 2 : 1>),  \
                         dim3((pairs + 7) / 8 * 8 * ((vts + 1) / 2)), block, 0, s, g); \
    else                                                                         \
      hipLaunchKernelGGL((recurrence_chain_kernel<E_, DELTA, 1>), chain, block,  \
                         0, s, g);                                               \
  } while (0)
  if (g.a.D <= 64) T5D_CH(1);
  else if (g.a.D <= 128) T5D_CH(2);
  else if (g.a.D <= 256) T5D_CH(4);
  else T5D_CH(8);
#undef T5D_CH
}

// Prepare and scan.
template <bool DELTA, typename T>
static void launch_token_by_token(hipStream_t s, const RecArgs& g) {
  const t5d_recurrence& a = g.a;
  const bool qkv = a.taps > 0 || a.unit;
  const int64_t units = (int64_t)g.b.M * ((qkv ? 2 * a.G + a.H : 0) + a.H);
  hipLaunchKernelGGL(recurrence_prepare_kernel<T>, dim3((unsigned)((units + 3) / 4)),
                     dim3(256), 0, s, g);
  if (qkv) {
    launch_scan<DELTA, float>(s, g, g.wq, g.wk, g.wv, a.G * a.D, a.G * a.D,
                              a.H * a.Dv, 1.f);
  } else {
    const T* p = reinterpret_cast<const T*>(a.proj);
    launch_scan<DELTA, T>(s, g, p + a.off_q, p + a.off_k, p + a.off_v, a.ld_proj,
                          a.ld_proj, a.ld_proj, a.q_scale);
  }
}

template <typename T>
static int run_portions(hipStream_t s, const RecArgs& g) {
  const t5d_recurrence& a = g.a;
  if (g.wchunk != nullptr) {
    if (a.delta) launch_chunks<true, T>(s, g);
    else launch_chunks<false, T>(s, g);
  } else if (a.delta) {
    launch_token_by_token<true, T>(s, g);
  } else {
    launch_token_by_token<false, T>(s, g);
  }
  T5D_CHECK_LAUNCH("recurrence (portions)");
  if (a.taps > 1) {
    hipLaunchKernelGGL(recurrence_conv_tail_kernel<T>,
                       dim3((g.C + 255) / 256, g.b.S), dim3(256), 0, s, g);
    T5D_CHECK_LAUNCH("recurrence (convolution tail)");
  }
  const int64_t heads = (int64_t)g.b.M * a.H;
  const bool vec = a.Dv % 4 == 0 && a.Dv <= 128 && a.ld_out % 4 == 0 &&
                   a.ld_low % 4 == 0 && a.off_low_gate % 4 == 0 &&
                   ((uintptr_t)a.out | (uintptr_t)a.low) % 16 == 0;
  if (vec)
    hipLaunchKernelGGL((recurrence_finish_kernel<T, true>),
                       dim3((unsigned)((heads + 7) / 8)), dim3(256), 0, s, g);
  else
    hipLaunchKernelGGL((recurrence_finish_kernel<T, false>),
                       dim3((unsigned)((heads + 3) / 4)), dim3(256), 0, s, g);
  T5D_CHECK_LAUNCH("recurrence (finish)");
  return T5D_OK;
}

static int64_t round4(int64_t n) { return (n + 3) / 4 * 4; }

// Floats of scratch of the un-chunked kernels.
static int64_t portion_floats(int64_t M, int H, int G, int D, int Dv) {
  return 2 * round4(M * G * D) + 2 * round4(M * H * Dv) + round4(M * H);
}

static int channel_pad(int D) {
  return D <= 64 ? 64 : D <= 128 ? 128 : D <= 256 ? 256 : 512;
}
static int64_t chunk_floats(int64_t M, int S, int H, int D, int Dv) {
  const ChunkLayout lay(channel_pad(D), (Dv + 15) / 16 * 16);
  return (int64_t)chunk_base(M, S) * H * (int64_t)lay.size();
}

// Portions from here on run in chunks.
constexpr int kChunkFrom = 24;

}  // namespace t5d

using namespace t5d;

extern "C" int64_t t5d_recurrence_workspace_bytes(int M, int S, int H, int G, int D,
                                                  int Dv) {
  if (M <= 0 || S < 0 || H <= 0 || G <= 0 || D <= 0 || Dv <= 0) return -1;
  return 4 * (portion_floats(M, H, G, D, Dv) +
              (S > 0 ? chunk_floats(M, S, H, D, Dv) : 0));
}

extern "C" int t5d_recurrence_run(void* stream, const t5d_recurrence* a,
                                  const t5d_ragged* b, int variant) {
  T5D_REQUIRE(a && b, T5D_EINVAL, "t5d_recurrence_run: null arguments");
  T5D_REQUIRE(a->dtype == T5D_F32 || a->dtype == T5D_BF16, T5D_EINVAL,
              "t5d_recurrence_run: dtype %d", a->dtype);
  T5D_REQUIRE(a->H > 0 && a->G > 0 && a->H % a->G == 0 && a->D > 0 && a->Dv > 0 &&
                  a->taps >= 0 && a->H <= 65535,
              T5D_EINVAL, "t5d_recurrence_run: H=%d G=%d D=%d Dv=%d taps=%d", a->H,
              a->G, a->D, a->Dv, a->taps);
  T5D_REQUIRE(a->D <= 512, T5D_ELIMIT, "t5d_recurrence_run: key size %d > 512",
              a->D);
  T5D_REQUIRE(a->proj && a->low && a->decay_bias && a->norm && a->state && a->out &&
                  (a->decay == T5D_DECAY_SIGMOID_POWER || a->A_log) &&
                  (a->taps == 0 || (a->conv && a->conv_ring)) && b->tok_pos &&
                  b->tok_seq && b->seq_off && b->seq_start && b->seq_slot,
              T5D_EINVAL, "t5d_recurrence_run: null buffer");
  T5D_REQUIRE(b->M > 0 && b->S > 0 && b->S <= 65535 && b->max_len > 0 &&
                  b->max_len <= b->M,
              T5D_EINVAL, "t5d_recurrence_run: M=%d S=%d max_len=%d", b->M, b->S,
              b->max_len);
  T5D_REQUIRE(variant >= 0 && variant <= 3, T5D_EINVAL,
              "t5d_recurrence_run: variant %d", variant);
  if (a->low_w != nullptr) {  // the columns that are read, of those that it has
    const int64_t z = a->off_z + (int64_t)a->H * a->D,
                  gate = a->off_low_gate + (int64_t)a->H * a->Dv;
    T5D_REQUIRE(a->off_low >= 0 && a->low_k > 0 &&
                    (int64_t)a->off_low + a->low_k <= a->ld_proj && a->off_z >= 0 &&
                    z <= a->low_n && (a->gate != T5D_GATE_SIGMOID_LOW ||
                                      (a->off_low_gate >= 0 && gate <= a->low_n)),
                T5D_EINVAL,
                "t5d_recurrence_run: low-rank inputs %d + %d of %d, columns from %d and %d "
                "of %d", a->off_low, a->low_k, a->ld_proj, a->off_z, a->off_low_gate,
                a->low_n);
  }
  RecArgs g;
  g.a = *a; g.b = *b; g.gate = tls_gate;
  g.C = 2 * a->G * a->D + a->H * a->Dv;
  const bool can_step = b->max_len == 1 && b->M == b->S && a->D <= 256 &&
                        a->Dv <= 256 && a->Dv % 4 == 0 &&
                        (uintptr_t)a->state % 16 == 0;
  T5D_REQUIRE(variant != 1 || can_step, T5D_EINVAL,
              "t5d_recurrence_run: variant 1 does not cover this call");
  hipStream_t s = as_stream(stream);
  const bool step = variant == 1 || (variant == 0 && can_step);
  if (a->low_w != nullptr && !(step && low_rides(*a, b->S))) {
    const char* in =
        (const char*)a->proj + (size_t)a->off_low * (a->dtype == T5D_F32 ? 4 : 2);
    const int rc = t5d_dense(stream, a->dtype, T5D_F32, in, a->ld_proj, a->low_w, a->low,
                             a->ld_low, a->low_n, b->M, a->low_k, a->low_n, T5D_EPI_NONE,
                             0.f, 0.f, 0.f);
    if (rc != T5D_OK) return rc;
    g.a.low_w = nullptr;
  }
  if (step) {
    g.wq = g.wk = g.wv = g.wbeta = g.wo = g.wchunk = nullptr;
    g.order = nullptr;
    g.chunks = 0;
    const bool bf16 = a->dtype == T5D_BF16;
    if (a->delta) {
      if (bf16) launch_step<true, bf16_t>(s, g);
      else launch_step<true, float>(s, g);
    } else {
      if (bf16) launch_step<false, bf16_t>(s, g);
      else launch_step<false, float>(s, g);
    }
    T5D_CHECK_LAUNCH("recurrence (step)");
    return T5D_OK;
  }
  T5D_REQUIRE(a->workspace && (uintptr_t)a->workspace % 16 == 0, T5D_EINVAL,
              "t5d_recurrence_run: portions need a 16-byte aligned workspace");
  float* w = (float*)a->workspace;
  const int64_t qk = round4((int64_t)b->M * a->G * a->D),
                hv = round4((int64_t)b->M * a->H * a->Dv);
  g.wq = w; g.wk = w + qk; g.wv = w + 2 * qk; g.wo = w + 2 * qk + hv;
  g.wbeta = w + 2 * qk + 2 * hv;
  // (in chunks q has no scratch of its own)
  g.order = b->S > 1 && b->S <= (int64_t)b->M * a->G * a->D ? (int32_t*)g.wq : nullptr;
  const int64_t plain = portion_floats(b->M, a->H, a->G, a->D, a->Dv);
  g.chunks = (b->max_len + kChunk - 1) / kChunk;
  const bool fits =
      a->taps <= kChunkTaps && a->Dv <= 512 &&
      a->workspace_bytes >=
      4 * (plain + chunk_floats(b->M, b->S, a->H, a->D, a->Dv));
  T5D_REQUIRE(a->workspace_bytes >= 4 * plain && (variant != 3 || fits), T5D_EINVAL,
              "t5d_recurrence_run: a workspace of %lld bytes",
              (long long)a->workspace_bytes);
  g.wchunk = variant == 3 || (variant == 0 && fits && b->max_len >= kChunkFrom)
                 ? w + plain : nullptr;
  return a->dtype == T5D_BF16 ? run_portions<bf16_t>(s, g) : run_portions<float>(s, g);
}
