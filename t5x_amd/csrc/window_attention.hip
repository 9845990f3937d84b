// Causal softmax attention over a sliding window (or everything before), with
// grouped key / value heads, per-head norms of queries and keys, a linear
// distance bias and a sink in the denominator — for sequences that are fed in
// portions of any length.
//
// Keys and values live in a ring per (slot, key/value head): position p of the
// slot's sequence is row p % ring.  A launch first writes the new positions,
// then every query reads the ring; the ring holds at least window - 1 + portion
// rows, so nothing a query of the portion needs has been overwritten, and rows
// left by an earlier sequence of the slot lie outside every mask.  Rows are
// padded with zeros to HP (32, 64, 128 or 256 elements), ring is a multiple of
// 64: a tile of 64 keys that starts at a multiple of 64 is consecutive memory.
//
// Three kernels attend:
//   * rows (bfloat16, portions): a tile is 128 (token, head of the group) pairs,
//     so grouped heads share the keys and values that a workgroup stages in LDS.
//     Scores are formed transposed, S^T = K Q^T: a lane then holds 4 consecutive
//     keys of ONE query, which is the operand order of the second product
//     O^T = V^T P^T up to a permutation of the keys that the V^T reads follow —
//     the weights never cross lanes.  They enter that product as two bfloat16
//     terms (value + remainder), which keeps them to 16 bits of mantissa.
//   * step (bfloat16, one new token per sequence): norms, the ring update and the
//     attention in one kernel, a workgroup per (sequence, key/value head, part of
//     the keys); scores on the matrix cores with the group's heads as the columns,
//     weights times values in float32 on the vector ALUs, wavefronts merged
//     through LDS, parts through a small second kernel.
//   * wave (float32, and sizes the other two do not cover): one wavefront per
//     (token, head), all in float32.
#include "common.h"
#include "gemm_tiles.h"

namespace t5d {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNoMax = -1e30f;  // running maximum before the first key

struct WinArgs {
  t5d_window_attention a;
  t5d_ragged b;
  int HP, gs, splits;
  int tiles;  // window_rows_kernel: tiles of rows of the longest portion
  int flat;   // ... and whether its grid has one dimension, or (tiles, S, G)
  float* parts;  // [S, G, splits, gs, HP + 2]
  const int32_t* gate;
  // window_rows_kernel over a span instead of rings: position first[s] + i of
  // portion s is row off[s] + i, rows ld_kv apart, a head's HP columns side by side
  const int32_t *span_off, *span_first;
  int ld_kv;
};

// ---- norms of the new queries and keys, ring update ------------------------------
// One wavefront per (token, head vector): H queries, G keys, G values.
template <typename T>
__global__ void __launch_bounds__(256)
window_append_kernel(WinArgs g) {
  T5D_GATED(g.gate);
  const t5d_window_attention& a = g.a;
  const int lane = threadIdx.x & 63;
  const int nvec = a.H + 2 * a.G;
  const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= (int64_t)g.b.M * nvec) return;
  const int m = unit / nvec, vec = unit % nvec;
  const int seq = g.b.tok_seq[m];
  const int row = g.b.tok_pos[m] % a.ring;
  const T* p = reinterpret_cast<const T*>(a.proj) + (size_t)m * a.ld_proj;
  T* dst;
  const float* w = nullptr;
  int n = a.D;
  if (vec < a.H) {
    p += a.off_q + vec * a.D;
    w = a.q_norm;
    dst = reinterpret_cast<T*>(a.q_rows) + ((size_t)m * a.H + vec) * g.HP;
  } else {
    const bool key = vec < a.H + a.G;
    const int h = vec - a.H - (key ? 0 : a.G);
    const size_t r =
        ((size_t)g.b.seq_slot[seq] * a.G + h) * a.ring + row;
    dst = reinterpret_cast<T*>(key ? a.key_ring : a.value_ring) + r * g.HP;
    if (key) w = a.k_norm; else n = a.Dv;
    p += key ? a.off_k + h * a.D : a.off_v + h * a.Dv;
  }
  float inv = 1.f;
  if (w != nullptr) {
    float ss = 0.f;
    for (int i = lane; i < n; i += 64) {
      const float v = to_f32<T>(p[i]);
      ss = fmaf(v, v, ss);
    }
    inv = 1.0f / sqrtf(wave_sum(ss) / (float)n + a.eps);
  }
  for (int i = lane; i < g.HP; i += 64) {
    float v = 0.f;
    if (i < n) {
      v = to_f32<T>(p[i]);
      if (w != nullptr) v = v * inv * w[i];
    }
    Act<T>::store(dst + i, v);
  }
}

// The same for bfloat16 rows of whole 16-byte pieces: HP / 8 lanes per vector.
__global__ void __launch_bounds__(256)
window_append_vec_kernel(WinArgs g) {
  T5D_GATED(g.gate);
  const t5d_window_attention& a = g.a;
  const int lpv = g.HP / 8;  // 4, 8, 16 or 32: a power of two
  const int nvec = a.H + 2 * a.G;
  const int64_t unit = (int64_t)blockIdx.x * (256 / lpv) + threadIdx.x / lpv;
  const bool on = unit < (int64_t)g.b.M * nvec;
  const int m = on ? unit / nvec : 0, vec = on ? unit % nvec : 0;
  const int c = 8 * (threadIdx.x % lpv);
  const bool query = vec < a.H, key = !query && vec < a.H + a.G;
  const int h = query ? vec : vec - a.H - (key ? 0 : a.G);
  const int n = query || key ? a.D : a.Dv;
  const bf16_t* p = reinterpret_cast<const bf16_t*>(a.proj) + (size_t)m * a.ld_proj +
                    (query ? a.off_q + h * a.D : key ? a.off_k + h * a.D
                                                     : a.off_v + h * a.Dv);
  const float* w = query ? a.q_norm : key ? a.k_norm : nullptr;
  uint4 v = make_uint4(0, 0, 0, 0);
  if (on && c < n) v = *reinterpret_cast<const uint4*>(p + c);
  if (w != nullptr) {
    float f[8];
    unpack16(v, f);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
    for (int step = 1; step < lpv; step *= 2) ss += __shfl_xor(ss, step, 64);
    const float inv = 1.0f / sqrtf(ss / (float)n + a.eps);
    if (c < n) {
      const float4 x = *reinterpret_cast<const float4*>(w + c);
      const float4 y = *reinterpret_cast<const float4*>(w + c + 4);
      v.x = pack_bf16x2(f[0] * inv * x.x, f[1] * inv * x.y);
      v.y = pack_bf16x2(f[2] * inv * x.z, f[3] * inv * x.w);
      v.z = pack_bf16x2(f[4] * inv * y.x, f[5] * inv * y.y);
      v.w = pack_bf16x2(f[6] * inv * y.z, f[7] * inv * y.w);
    }
  }
  if (!on) return;
  bf16_t* dst;
  if (query) {
    dst = reinterpret_cast<bf16_t*>(a.q_rows) + ((size_t)m * a.H + h) * g.HP;
  } else {
    const size_t r = ((size_t)g.b.seq_slot[g.b.tok_seq[m]] * a.G + h) * a.ring +
                     g.b.tok_pos[m] % a.ring;
    dst = reinterpret_cast<bf16_t*>(key ? a.key_ring : a.value_ring) + r * g.HP;
  }
  *reinterpret_cast<uint4*>(dst + c) = v;
}

// ---- float32 / any size -----------------------------------------------------------
template <typename T, int NV>
__global__ void __launch_bounds__(64)
window_wave_kernel(WinArgs g) {
  T5D_GATED(g.gate);
  const t5d_window_attention& a = g.a;
  extern __shared__ float lds[];
  float* s_q = lds;           // [HP]
  float* s_p = lds + g.HP;    // [64]
  const int lane = threadIdx.x;
  const int m = blockIdx.x, h = blockIdx.y, kv = h / g.gs;
  const int seq = g.b.tok_seq[m], i = g.b.tok_pos[m];
  const size_t base = ((size_t)g.b.seq_slot[seq] * a.G + kv) * a.ring;
  const T* K = reinterpret_cast<const T*>(a.key_ring) + base * g.HP;
  const T* V = reinterpret_cast<const T*>(a.value_ring) + base * g.HP;
  const T* q = reinterpret_cast<const T*>(a.q_rows) + ((size_t)m * a.H + h) * g.HP;
  for (int d = lane; d < g.HP; d += 64) s_q[d] = to_f32<T>(q[d]);
  __syncthreads();
  const float slope = a.slopes != nullptr ? a.slopes[h] : 0.f;
  float mx = kNoMax, l = 0.f;
  if (a.sink != nullptr) {
    mx = a.sink[h] * kLog2e;
    l = 1.f;
  }
  float acc[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) acc[n] = 0.f;
  const int lo = a.window > 0 ? max(0, i - a.window + 1) : 0;
  for (int j0 = lo; j0 <= i; j0 += 64) {
    const int j = j0 + lane;
    float s = -INFINITY;
    if (j <= i) {
      const T* k = K + (size_t)(j % a.ring) * g.HP;
      float dot = 0.f;
      constexpr int E = Act<T>::kElemsPer16B;
      for (int d = 0; d < g.HP; d += E) {
        float f[E];
        unpack16(*reinterpret_cast<const uint4*>(k + d), f);
#pragma unroll
        for (int e = 0; e < E; ++e) dot = fmaf(f[e], s_q[d + e], dot);
      }
      s = (dot * a.scale - slope * (float)(i - j)) * kLog2e;
    }
    const float top = fmaxf(mx, wave_max(s));
    const float alpha = exp2f(mx - top);
    const float p = exp2f(s - top);
    mx = top;
    l = l * alpha + wave_sum(p);
    __syncthreads();
    s_p[lane] = p;
    __syncthreads();
    const int cnt = min(64, i - j0 + 1);
#pragma unroll
    for (int n = 0; n < NV; ++n) acc[n] *= alpha;
    for (int jj = 0; jj < cnt; ++jj) {
      const T* v = V + (size_t)((j0 + jj) % a.ring) * g.HP;
      const float w = s_p[jj];
#pragma unroll
      for (int n = 0; n < NV; ++n)
        if (lane + 64 * n < a.Dv) acc[n] = fmaf(w, to_f32<T>(v[lane + 64 * n]), acc[n]);
    }
  }
  T* o = reinterpret_cast<T*>(a.out) + (size_t)m * a.ld_out + (size_t)h * a.Dv;
#pragma unroll
  for (int n = 0; n < NV; ++n)
    if (lane + 64 * n < a.Dv) Act<T>::store(o + lane + 64 * n, acc[n] / l);
}

// ---- portions, bfloat16 -------------------------------------------------------------
__device__ __forceinline__ f32x4_v mfma(const Frag& x, const Frag& y, f32x4_v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, y.v, c, 0, 0, 0);
}

typedef __attribute__((address_space(3))) void* lds_void_t;
typedef __attribute__((address_space(1))) const void* glb_void_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4_v;
typedef __attribute__((address_space(3))) s16x4_v* lds_s16x4_t;

// A running maximum is raised, and what has been summed rescaled, only when a
// score passes it by this much (in powers of two): weights then reach 2^8, which
// their two terms and the float32 sums hold as well as weights up to 1.
constexpr float kMaxSlack = 8.0f;

// Keys and values of 64 positions at a time go from memory straight into LDS (no
// staging registers), one tile ahead in a second pair of buffers, one barrier per
// tile.  Rows lie in LDS as they are; the 16-byte pieces of a row are exchanged by
// an XOR with its number, which each lane applies to the address it fetches, so
// that 16 rows of one piece (key operands) and 8 rows of one 32-byte pair (value
// operands) cover all banks.  The operands of V^T are read with the transposing
// LDS read: 16 lanes give it 4 keys x 16 dims and get 4 keys of a dim each.
// BIAS: with slopes, or a scale that is not positive.
// Per tile and wavefront 96 matrix instructions (1536 cycles) stand against ~390
// vector instructions (1950 cycles with the 32 exponentials): what bounds the kernel
// is that the two hardly overlap at two wavefronts per SIMD (38 % and 43 % busy by the
// counters, no bank conflicts).  Measured, heads of 128 over 1024
// positions, 4 x 4096 tokens: 8 heads over 2 key/value heads 206 -> 115 us, 8 heads
// over expanded latents in pieces of 2048 118 -> 60 us each.  The kernel before
// staged tiles through registers, with a second barrier and V transposed on the way
// by 4-byte stores, masked every tile and rescaled in every tile.
template <int DT, bool SPAN, bool BIAS>
__global__ void __launch_bounds__(256, DT <= 4 ? 2 : 1)
window_rows_kernel(WinArgs g) {
  constexpr int HP = DT * 32, VT = DT * 2, KB = 64, MT = 2;
  constexpr int PP = HP / 8;  // 16-byte pieces per row
  // buffers of their own, so that the compiler can tell a read of one tile from a
  // load of the next
  __shared__ uint4 s_k0[KB * PP], s_v0[KB * PP], s_k1[KB * PP], s_v1[KB * PP];
  T5D_GATED(g.gate);
  const t5d_window_attention& a = g.a;
  // The tiles of one (portion, key/value head) read the same keys and values:
  // consecutive block ids go round-robin over the 8 XCDs, so theirs are 8 apart.
  const int gs = g.gs;
  int seq = blockIdx.y, kv = blockIdx.z, nth = blockIdx.x;
  bool turn = false;
  if (g.flat) {
    const int pair = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / g.tiles);
    if (pair >= a.G * g.b.S) return;
    seq = pair / a.G;
    kv = pair - seq * a.G;
    nth = (int)(blockIdx.x >> 3) % g.tiles;
    turn = (pair >> 3) * g.tiles / 32 % 2 != 0;
  }
  const int off = g.b.seq_off[seq];
  const int rows = (g.b.seq_off[seq + 1] - off) * gs;
  // Long tiles first, where the next 256 blocks begin the other way round (turn): the
  // two tiles of a CU are then a long one and a short one.
  const int r0 = (turn ? nth : g.tiles - 1 - nth) * (64 * MT);
  if (r0 >= rows) return;
  const int start = g.b.seq_start[seq];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, gq = lane >> 4;
  const int W = a.window > 0 ? a.window : (1 << 30);
  const size_t base = SPAN ? (size_t)g.span_off[seq] * g.ld_kv + (size_t)kv * HP
                           : ((size_t)g.b.seq_slot[seq] * a.G + kv) * a.ring * HP;
  const bf16_t* K = reinterpret_cast<const bf16_t*>(a.key_ring) + base;
  const bf16_t* V = reinterpret_cast<const bf16_t*>(a.value_ring) + base;
  const int ld_kv = SPAN ? g.ld_kv : HP;
  const int first = SPAN ? g.span_first[seq] : 0;

  const float scale2 = a.scale * kLog2e;
  int pos[MT], tok[MT], head[MT];
  float slope2[MT], mx[MT], l[MT];
  Frag qf[MT][DT];
  const int rw = r0 + wave * 16 * MT;  // the wavefront's first row
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = min(rw + 16 * mt + n16, rows - 1);  // past the end: not stored
    const int t = r / gs;
    head[mt] = kv * gs + (r - t * gs);
    tok[mt] = off + t;
    pos[mt] = start + t;
    slope2[mt] = BIAS && a.slopes != nullptr ? a.slopes[head[mt]] * kLog2e : 0.f;
    mx[mt] = a.sink != nullptr ? a.sink[head[mt]] * kLog2e : kNoMax;
    l[mt] = a.sink != nullptr && gq == 0 ? 1.f : 0.f;
    const bf16_t* q = reinterpret_cast<const bf16_t*>(a.q_rows) +
                      ((size_t)tok[mt] * a.H + head[mt]) * HP + 8 * gq;
#pragma unroll
    for (int kk = 0; kk < DT; ++kk)
      qf[mt][kk].u = *reinterpret_cast<const uint4*>(q + 32 * kk);
  }
  f32x4_v o[VT][MT];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) o[vt][mt] = (f32x4_v){0.f, 0.f, 0.f, 0.f};

  const int i_lo = start + r0 / gs;
  const int i_hi = start + min(r0 + 64 * MT - 1, rows - 1) / gs;
  const bool wave_on = rw < rows;
  const int wi_lo = start + min(rw, rows - 1) / gs;
  const int wi_hi = start + min(rw + 16 * MT - 1, rows - 1) / gs;
  const int j_begin = max(0, i_lo - W + 1) & ~(KB - 1);

  // what to exchange the pieces of a row by: keys, then pairs of values
  const auto k_swap = [](int row) {
    return PP >= 16 ? row & 15 : (row / (16 / PP)) & (PP - 1);
  };
  const auto v_swap = [](int row) {
    return PP >= 16 ? row & 7 : (row / (16 / PP)) & (PP / 2 - 1);
  };
  int k_off[DT], v_off[DT];  // of the pieces this lane fetches
#pragma unroll
  for (int i = 0; i < DT; ++i) {
    const int f = (wave * DT + i) * 64 + lane, row = f / PP, piece = f % PP;
    k_off[i] = row * ld_kv + 8 * (piece ^ k_swap(row));
    v_off[i] = row * ld_kv + 8 * (piece ^ (2 * v_swap(row)));
  }
  const auto fetch = [&](int jt, uint4* sk, uint4* sv) {
    const size_t r = (size_t)(SPAN ? jt - first : jt % a.ring) * ld_kv;
#pragma unroll
    for (int i = 0; i < DT; ++i)
      __builtin_amdgcn_global_load_lds((glb_void_t)(K + r + k_off[i]),
                                       (lds_void_t)(sk + (wave * DT + i) * 64), 16, 0,
                                       0);
#pragma unroll
    for (int i = 0; i < DT; ++i)
      __builtin_amdgcn_global_load_lds((glb_void_t)(V + r + v_off[i]),
                                       (lds_void_t)(sv + (wave * DT + i) * 64), 16, 0,
                                       0);
  };
  const int k_row = n16 * PP, k_x = k_swap(n16);
  const int v_key = 4 * gq + (n16 >> 2);
  const int v_at = v_key * PP * 16 + 8 * (n16 & 3), v_x = 32 * v_swap(v_key);
  const auto attend = [&](int jt, const uint4* sk, const uint4* sv) {
    if (!wave_on || jt > wi_hi || jt + KB - 1 <= wi_lo - W) return;
    f32x4_v s[4][MT];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) s[t][mt] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
    // Operands are read one group ahead of the products that take them; the fences
    // keep the compiler from reading each group when it is due.
    Frag kf[2][4];
    const auto keys = [&](int kk) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        kf[kk & 1][t].u = sk[16 * t * PP + k_row + ((4 * kk + gq) ^ k_x)];
    };
    keys(0);
#pragma unroll
    for (int kk = 0; kk < DT; ++kk) {
      if (kk + 1 < DT) keys(kk + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          s[t][mt] = mfma(kf[kk & 1][t], qf[mt][kk], s[t][mt]);
    }
    // V^T of dims 32 (n % (VT / 2)) .. + 31 and keys 32 (n / (VT / 2)) .. + 31
    constexpr int NV = VT / 2;
    Frag vf[2][2];
    const auto values = [&](int n) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const char* v = reinterpret_cast<const char*>(sv) + 32 * (n / NV) * PP * 16 +
                        v_at + ((32 * (2 * (n % NV) + j)) ^ v_x);
        union { s16x4_v h[2]; Frag f; } x;
        x.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)v);
        x.h[1] =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(v + 16 * PP * 16));
        vf[n & 1][j] = x.f;
      }
    };
    const bool edge = !(jt + KB - 1 <= wi_lo && jt > wi_hi - W);
    float top[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int d0 = pos[mt] - jt - 4 * gq;  // distance to this lane's first key
      if constexpr (BIAS) {
        const float far = -slope2[mt] * (float)d0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            s[t][mt][i] = fmaf(s[t][mt][i], scale2,
                               fmaf(slope2[mt], (float)(16 * t + i), far));
      }
      if (edge) {
        asm volatile("");  // (a branch: the compiler would select in every tile)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            s[t][mt][i] = (uint32_t)(d0 - 16 * t - i) < (uint32_t)W ? s[t][mt][i]
                                                                    : -INFINITY;
      }
      top[mt] = -INFINITY;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) top[mt] = fmaxf(top[mt], s[t][mt][i]);
      top[mt] = rows_max(top[mt]) * (BIAS ? 1.f : scale2);
    }
    bool raise = false;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) raise |= top[mt] > mx[mt] + kMaxSlack;
    if (__builtin_amdgcn_ballot_w64(raise) != 0) {
      asm volatile("");
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float to = fmaxf(mx[mt], top[mt]);
        const float alpha = __builtin_amdgcn_exp2f(mx[mt] - to);
        mx[mt] = to;
        l[mt] *= alpha;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[vt][mt][i] *= alpha;
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(
              BIAS ? s[t][mt][i] - mx[mt] : fmaf(s[t][mt][i], scale2, -mx[mt]));
          s[t][mt][i] = p;
          sum += p;
        }
      l[mt] += sum;
    }
    values(0);
    // weights of keys {16 (2 kb) + 4 gq + 0..3, 16 (2 kb + 1) + 4 gq + 0..3}
    Frag hi[2][MT], lo[2][MT];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        uint32_t h[4], r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = s[2 * kb + (e >> 1)][mt][2 * (e & 1)];
          const float p1 = s[2 * kb + (e >> 1)][mt][2 * (e & 1) + 1];
          h[e] = pack_bf16x2(p0, p1);
          r[e] = pack_bf16x2(p0 - bf16lo_to_f32(h[e]), p1 - bf16hi_to_f32(h[e]));
        }
        hi[kb][mt].u = make_uint4(h[0], h[1], h[2], h[3]);
        lo[kb][mt].u = make_uint4(r[0], r[1], r[2], r[3]);
      }
#pragma unroll
    for (int n = 0; n < 2 * NV; ++n) {
      if (n + 1 < 2 * NV) values(n + 1);
      __builtin_amdgcn_sched_barrier(0);
      // (four products between two that add to the same tile)
      const int kb = n / NV, vt = 2 * (n % NV);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          o[vt + j][mt] = mfma(vf[n & 1][j], hi[kb][mt], o[vt + j][mt]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          o[vt + j][mt] = mfma(vf[n & 1][j], lo[kb][mt], o[vt + j][mt]);
    }
  };
  // All my loads have landed and my reads of the other tile have returned; behind
  // the barrier everyone's have.
  const auto meet = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch(j_begin, s_k0, s_v0);
  for (int jt = j_begin; jt <= i_hi; jt += 2 * KB) {
    meet();
    if (jt + KB <= i_hi) fetch(jt + KB, s_k1, s_v1);
    attend(jt, s_k0, s_v0);
    if (jt + KB > i_hi) break;
    meet();
    if (jt + 2 * KB <= i_hi) fetch(jt + 2 * KB, s_k0, s_v0);
    attend(jt + KB, s_k1, s_v1);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const float inv = 1.0f / rows_sum(l[mt]);
    if (rw + 16 * mt + n16 >= rows) continue;
    bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + (size_t)tok[mt] * a.ld_out +
                  (size_t)head[mt] * a.Dv;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const int d = 16 * vt + 4 * gq;
      if ((a.Dv & 3) == 0) {
        if (d < a.Dv)
          *reinterpret_cast<uint2*>(out + d) =
              make_uint2(pack_bf16x2(o[vt][mt][0] * inv, o[vt][mt][1] * inv),
                         pack_bf16x2(o[vt][mt][2] * inv, o[vt][mt][3] * inv));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (d + i < a.Dv) out[d + i] = f32_to_bf16(o[vt][mt][i] * inv);
      }
    }
  }
}

// ---- one new token per sequence, bfloat16 ----------------------------------------------
__device__ __forceinline__ void wave_lds_fence() {
  // LDS operations of a wavefront complete in order; this only keeps the
  // compiler from moving one lane's read above another lane's write.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// (Heads of 129 to 256, a key head per query head: 268 registers as the compiler would
// have it, 250 and a second workgroup per CU when asked to.  us, 268 / 250: 128 rows of 4
// heads of 256, window 512 61.2 / 56.3; 64 of 8 heads of 200, window 1024 105 / 101.)
template <int DT, int GS>
__global__ void __launch_bounds__(256, DT == 8 && GS == 1 ? 2 : 1)
window_step_kernel(WinArgs g) {
  constexpr int HP = DT * 32;
  constexpr int QS = HP + 8;
  constexpr int LPR = HP / 8;       // lanes on one value row
  constexpr int KPI = 64 / LPR;     // keys per value load
  constexpr int VL = 64 / KPI;      // value loads of a tile
  constexpr int VR = VL < 8 ? VL : 8;  // of them ahead (registers)
  __shared__ __align__(16) bf16_t s_q[16 * QS];
  __shared__ __align__(16) bf16_t s_new[2][HP];  // the new key and value
  __shared__ __align__(16) float s_w[4][64 * GS];  // weights [key][head]
  __shared__ float s_alpha[4][16];
  __shared__ float s_m[4][16], s_l[4][16];
  __shared__ __align__(16) float s_o[4][GS * HP];
  T5D_GATE_READ(g.gate);
  const t5d_window_attention& a = g.a;
  const int seq = blockIdx.x / a.G, kv = blockIdx.x % a.G, part = blockIdx.y;
  const int gs = g.gs;              // <= GS
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, gq = lane >> 4;
  const int W = a.window > 0 ? a.window : (1 << 30);

  // The group's queries (the last one again up to GS), the new key and value: vectors
  // 0 .. GS - 1, GS, GS + 1.  They depend on nothing but the arguments and are requested
  // first, the flag and the sequence's place with them.
  constexpr int U = (HP + 63) / 64, NV = (GS + 5) / 4;  // vectors wave, wave + 4, ...
  bf16_t raw[NV][U];
  float scale[NV][U];
  const auto width = [&](int vec) { return vec > GS ? a.Dv : a.D; };
  const auto norm = [&](int vec) {
    return vec < GS ? a.q_norm : vec == GS ? a.k_norm : nullptr;
  };
  const bf16_t* p = reinterpret_cast<const bf16_t*>(a.proj) + (size_t)seq * a.ld_proj;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int vec = min(wave + 4 * v, GS + 1);
    const bf16_t* src = p + (vec < GS ? a.off_q + (kv * gs + min(vec, gs - 1)) * a.D
                             : vec == GS ? a.off_k + kv * a.D
                                         : a.off_v + kv * a.Dv);
    const float* w = norm(vec);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int d = min(lane + 64 * u, width(vec) - 1);
      raw[v][u] = src[d];
      scale[v][u] = w != nullptr ? w[d] : 1.f;
    }
  }
  const int i = g.b.seq_start[seq];
  const size_t base = ((size_t)g.b.seq_slot[seq] * a.G + kv) * a.ring;
  T5D_GATE_TEST();
  bf16_t* K = reinterpret_cast<bf16_t*>(a.key_ring) + base * HP;
  bf16_t* V = reinterpret_cast<bf16_t*>(a.value_ring) + base * HP;

  // The keys and (the first) values of this wavefront's next 64 positions.
  const int j_begin = max(0, i - W + 1) & ~63;
  const int vsub = lane / LPR, vpiece = lane % LPR;
  Frag kf[4][DT];
  uint4 vr[VR];
  const auto request_tile = [&](int jt) {
    const size_t r = (size_t)(jt % a.ring);
    const bf16_t* kt = K + r * HP;
    const bf16_t* vt = V + r * HP;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int kk = 0; kk < DT; ++kk)
        kf[t][kk].u = *reinterpret_cast<const uint4*>(
            kt + (size_t)(16 * t + n16) * HP + 32 * kk + 8 * gq);
#pragma unroll
    for (int u = 0; u < VR; ++u)
      vr[u] = *reinterpret_cast<const uint4*>(
          vt + (size_t)(u * KPI + vsub) * HP + 8 * vpiece);
  };

  // The queries, the new key and value -> LDS.  (Rows GS .. 15 of the query tile are
  // whatever is there: columns of the products that nothing looks at.)  All of a
  // wavefront's vectors and its first tile are requested before the first is looked at;
  // the tile that holds the new row's place does not wait for the ring: it gets the new
  // key, and the new value is added at the end.  The ring takes both from the one
  // wavefront that has this tile, when it is done with it: what the tile read there,
  // weighed by zero, is what the ring held before and nothing that is just being written.
  // One row of 8 heads over 2 with a window of 1024: 15.5 us one after the other and the
  // tile behind the barrier, 13.1 with the tile of the new row only behind it, 11.0 so
  // and with a third fewer instructions; with the kernel that merges the parts, for 1 x
  // (16 over 4), 4 x (8 over 2) of 300 positions, 64 x (8 over 2), 256 x (8 over 2): 16.5
  // -> 12.2, 13.4 -> 10.7, 23.6 -> 22.7, 54 -> 52.8.
  const int jt0 = j_begin + 64 * (part + g.splits * wave);
  {
    if (jt0 <= i) request_tile(jt0);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int vec = min(wave + 4 * v, GS + 1);
      const int n = width(vec);
      const bool normed = norm(vec) != nullptr;
      float f[U];
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        f[u] = lane + 64 * u < n ? bf16_to_f32(raw[v][u]) : 0.f;
        ss = fmaf(f[u], f[u], ss);
      }
      const float inv = normed ? 1.0f / sqrtf(wave_sum(ss) / (float)n + a.eps) : 1.f;
      bf16_t* dst = vec < GS ? s_q + vec * QS : s_new[vec - GS];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int d = lane + 64 * u;
        if (d < HP) dst[d] = f32_to_bf16(f[u] * inv * scale[v][u]);
      }
    }
  }
  // (what goes to and comes from memory is not waited for)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  Frag qf[DT];
#pragma unroll
  for (int kk = 0; kk < DT; ++kk)
    qf[kk].u = *reinterpret_cast<const uint4*>(s_q + n16 * QS + 32 * kk + 8 * gq);
  const int head = kv * gs + min(n16, gs - 1);
  const float scale2 = a.scale * kLog2e;
  const float slope2 = a.slopes != nullptr ? a.slopes[head] * kLog2e : 0.f;
  float mx = kNoMax, l = 0.f;
  float acc[GS][8], w_new[GS];
  bool holds_new = false;  // this wavefront's last tile is the new row's
#pragma unroll
  for (int h = 0; h < GS; ++h) {
    w_new[h] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[h][e] = 0.f;
  }

  for (int jt = jt0; jt <= i; jt += 64 * 4 * g.splits) {
    const bf16_t* vt = V + (size_t)(jt % a.ring) * HP;
    if (jt != jt0) request_tile(jt);
    if (jt + 63 >= i) {  // the new row's place is in this tile
      const int r = i - jt;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (16 * t + n16 == r) {
#pragma unroll
          for (int kk = 0; kk < DT; ++kk)
            kf[t][kk].u = *reinterpret_cast<const uint4*>(s_new[0] + 32 * kk + 8 * gq);
        }
    }
    f32x4_v s[4];
    float top = mx;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      s[t] = (f32x4_v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < DT; ++kk) s[t] = mfma(kf[t][kk], qf[kk], s[t]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int dist = i - jt - 16 * t - 4 * gq - e;
        const float v = fmaf(s[t][e], scale2, -slope2 * (float)dist);
        s[t][e] = dist >= 0 && dist < W ? v : -INFINITY;
        top = fmaxf(top, s[t][e]);
      }
    top = rows_max(top);
    const float alpha = __builtin_amdgcn_exp2f(mx - top);
    mx = top;
    float sum = 0.f;
    wave_lds_fence();  // the previous tile's weights have been read
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p = __builtin_amdgcn_exp2f(s[t][e] - top);
        sum += p;
        if (n16 < GS) s_w[wave][(16 * t + 4 * gq + e) * GS + n16] = p;
      }
    l = l * alpha + sum;
    if (gq == 0) s_alpha[wave][n16] = alpha;
    wave_lds_fence();
    if (jt + 63 >= i) {  // the new value is added at the end (this is the last tile)
      holds_new = true;
      float* w = &s_w[wave][(i - jt) * GS];
#pragma unroll
      for (int h = 0; h < GS; ++h) w_new[h] = w[h];
      asm volatile("" ::: "memory");  // (an order for the compiler; no wait, see above)
      if (lane < GS) w[lane] = 0.f;
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int h = 0; h < GS; ++h) {
      const float al = s_alpha[wave][h];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[h][e] *= al;
    }
#pragma unroll
    for (int u0 = 0; u0 < VL; u0 += VR) {
      if (u0 > 0) {
#pragma unroll
        for (int u = 0; u < VR; ++u)
          vr[u] = *reinterpret_cast<const uint4*>(
              vt + (size_t)((u0 + u) * KPI + vsub) * HP + 8 * vpiece);
      }
#pragma unroll
      for (int u = 0; u < VR; ++u) {
        float f[8];
        unpack16(vr[u], f);
        const float* w = &s_w[wave][((u0 + u) * KPI + vsub) * GS];
#pragma unroll
        for (int h = 0; h < GS; ++h) {
          const float p = w[h];
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[h][e] = fmaf(p, f[e], acc[h][e]);
        }
      }
    }
  }
  if (holds_new) {  // (element by element: a ring may start anywhere)
    const size_t row = (size_t)(i % a.ring) * HP;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int d = lane + 64 * u;
      if (d < HP) {
        K[row + d] = s_new[0][d];
        V[row + d] = s_new[1][d];
      }
    }
  }
  // (the new value, by the wavefront that has its weight alone: it may be infinite, and
  // nothing times that is not nothing)
  if (holds_new && vsub == 0) {
    float f[8];
    unpack16(*reinterpret_cast<const uint4*>(s_new[1] + 8 * vpiece), f);
#pragma unroll
    for (int h = 0; h < GS; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[h][e] = fmaf(w_new[h], f[e], acc[h][e]);
  }
  // Sum over the lanes that took other keys of the same value piece, then the
  // wavefronts' results meet in LDS.
#pragma unroll
  for (int h = 0; h < GS; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float v = acc[h][e];
      if (LPR <= 4) v += lane_xor4(v);
      if (LPR <= 8) v += lane_xor8(v);
      if (LPR <= 16) {
        v = rows_sum(v);
      } else {
        const auto w = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(w[0]) + __uint_as_float(w[1]);
      }
      acc[h][e] = v;
    }
  if (vsub == 0) {
#pragma unroll
    for (int h = 0; h < GS; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) s_o[wave][h * HP + 8 * vpiece + e] = acc[h][e];
  }
  const float lt = rows_sum(l);
  if (gq == 0) {
    s_m[wave][n16] = mx;
    s_l[wave][n16] = lt;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < gs * HP; e += 256) {
    const int h = e / HP, d = e - h * HP;
    if (d >= a.Dv) continue;
    float top = fmaxf(fmaxf(s_m[0][h], s_m[1][h]), fmaxf(s_m[2][h], s_m[3][h]));
    const bool last = g.splits == 1;
    const float sink2 = last && a.sink != nullptr ? a.sink[kv * gs + h] * kLog2e : kNoMax;
    top = fmaxf(top, sink2);
    float num = 0.f, den = last && a.sink != nullptr ? exp2f(sink2 - top) : 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float c = exp2f(s_m[w][h] - top);
      num = fmaf(c, s_o[w][e], num);
      den = fmaf(c, s_l[w][h], den);
    }
    if (last) {
      reinterpret_cast<bf16_t*>(a.out)[(size_t)seq * a.ld_out +
                                       (size_t)(kv * gs + h) * a.Dv + d] =
          f32_to_bf16(num / den);
    } else {
      float* o = g.parts + (((size_t)blockIdx.x * g.splits + part) * gs + h) * (HP + 2);
      o[d] = num;
      if (d == 0) {
        o[HP] = top;
        o[HP + 1] = den;
      }
    }
  }
}

constexpr int kMaxSplits = 16;

// The parts of window_step_kernel: one wavefront per (sequence, head).  Lane s looks at
// the maximum and the sum of part s; the parts' rows are requested with them (a loop
// over the parts, one wait each, three times over: 5.0 us for 64 rows of 8 heads and two
// parts, now 4.6; 8 rows of 32 heads, 16 parts, with the kernel in front 26.0 -> 17.9).
__global__ void __launch_bounds__(64)
window_merge_kernel(WinArgs g) {
  T5D_GATE_READ(g.gate);
  const t5d_window_attention& a = g.a;
  const int seq = blockIdx.x / a.H, h = blockIdx.x % a.H;
  const int kv = h / g.gs, hh = h % g.gs;
  const int step = g.gs * (g.HP + 2);
  const float* p = g.parts + ((size_t)seq * a.G + kv) * g.splits * step +
                   (size_t)hh * (g.HP + 2);
  const int lane = threadIdx.x, mine = min(lane & 15, g.splits - 1);
  const float part_top = p[mine * step + g.HP];
  const float part_den = p[mine * step + g.HP + 1];
  const float sink2 = a.sink != nullptr ? a.sink[h] * kLog2e : kNoMax;
  float row[kMaxSplits];
  const auto request = [&](int d) {
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s)
      if (s < g.splits) row[s] = p[s * step + d];
  };
  request(min(lane, a.Dv - 1));
  T5D_GATE_TEST();
  const float top = fmaxf(lanes16_max(part_top), sink2);
  const float weight = exp2f(part_top - top);
  float c[kMaxSplits];
  float den = a.sink != nullptr ? exp2f(sink2 - top) : 0.f;
#pragma unroll
  for (int s = 0; s < kMaxSplits; ++s) {
    c[s] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), s));
    if (s < g.splits)
      den = fmaf(c[s],
                 __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(part_den), s)),
                 den);
  }
  for (int d = lane; d < a.Dv; d += 64) {
    if (d >= 64) request(d);
    float num = 0.f;
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s)
      if (s < g.splits) num = fmaf(c[s], row[s], num);
    reinterpret_cast<bf16_t*>(a.out)[(size_t)seq * a.ld_out + (size_t)h * a.Dv + d] =
        f32_to_bf16(num / den);
  }
}

static int step_splits(const t5d_window_attention& a, int S) {
  const int span = a.window > 0 ? min(a.window, a.ring) : a.ring;
  int n = 1;
  while (n < kMaxSplits && S * a.G * n < 256 && span >= 512 * n) n *= 2;
  // Where there are parts to be merged anyhow: one tile of 64 positions per wavefront
  // while CUs are left.  A window of 1024 touches 17 tiles, the last of which made one of
  // 16 wavefronts walk two.  (Two parts for the fifth tile of a window of 256, 1 row of 8
  // heads over 2: 11.1 us as one part does, over 100 positions 10.3 against 8.1; 64 rows
  // 13.5 against 12.7.)
  while (n > 1 && n < kMaxSplits && 4 * n < span / 64 + 1 && S * a.G * (n + 1) <= 256) ++n;
  return n;
}

// The step kernel's template sizes: heads per group rounded up, 0 if it does
// not cover the shape.
static int step_group(int gs, int HP) {
  if (HP > 256 || gs > 16) return 0;
  int n = 1;
  while (n < gs) n *= 2;
  return n * HP <= 2048 ? n : 0;
}

template <typename T>
static void launch_wave(hipStream_t s, const WinArgs& g) {
  const int nv = (g.a.Dv + 63) / 64;
  const dim3 grid(g.b.M, g.a.H), block(64);
  const size_t lds = (g.HP + 64) * sizeof(float);
#define T5D_WW(N_) \
  hipLaunchKernelGGL((window_wave_kernel<T, N_>), grid, block, lds, s, g)
  if (nv <= 1) T5D_WW(1);
  else if (nv <= 2) T5D_WW(2);
  else if (nv <= 4) T5D_WW(4);
  else T5D_WW(16);
#undef T5D_WW
}

static WinArgs win_args(const t5d_window_attention& a, const t5d_ragged& b, int HP) {
  WinArgs g = {};
  g.a = a; g.b = b;
  g.HP = HP; g.gs = a.H / a.G; g.splits = 1;
  g.parts = (float*)a.workspace;
  g.gate = tls_gate;
  return g;
}

template <bool SPAN>
static void launch_rows_tiles(hipStream_t s, WinArgs g) {
  g.tiles = ((int64_t)g.b.max_len * g.gs + 127) / 128;
  const int64_t pairs = (int64_t)g.b.S * g.a.G;
  // The one-dimensional grid keeps the tiles of a pair on one XCD, whose 32 CUs then
  // share its keys and values: 3 to 20 % faster where every XCD gets about the same
  // (heads of 128, 3000 tokens x 4 heads, us with it / without: 8 pairs 98 / 109, 16 172
  // / 185, 32 309 / 333; heads of 200: 297 / 367, 545 / 711, 1116 / 1373).  Few pairs
  // leave XCDs idle (1 pair 79 / 40, 2 85 / 47, 4 90 / 67, 6 93 / 94, 9 144 / 119, 12
  // 150 / 150, 17 216 / 200; heads of 200, 1 pair 269 / 120), unless an XCD has a CU for
  // each tile (heads of 64, 1500 tokens, 9 pairs: 31.8 / 33.7).  And a dimension of a
  // grid holds fewer than 2^32 threads: many portions beside one of very many
  // (token, head) pairs take three.
  const int64_t turns = (pairs + 7) / 8, blocks = turns * 8 * g.tiles;
  g.flat = blocks < (1LL << 24) && (turns * g.tiles <= 32 || turns * 24 <= pairs * 4);
  const dim3 grid = g.flat ? dim3((unsigned)blocks) : dim3(g.tiles, g.b.S, g.a.G);
  const dim3 block(256);
#define T5D_ROWS(DT_)                                                              \
  do {                                                                             \
    if (g.a.slopes != nullptr || !(g.a.scale > 0.f))                               \
      hipLaunchKernelGGL((window_rows_kernel<DT_, SPAN, true>), grid, block, 0, s, g); \
    else                                                                           \
      hipLaunchKernelGGL((window_rows_kernel<DT_, SPAN, false>), grid, block, 0, s, g); \
  } while (0)
  if (g.HP == 32) T5D_ROWS(1);
  else if (g.HP == 64) T5D_ROWS(2);
  else if (g.HP == 128) T5D_ROWS(4);
  else T5D_ROWS(8);
#undef T5D_ROWS
}

int launch_window_span(hipStream_t s, const t5d_window_attention& a,
                       const t5d_ragged& b, const t5d_span& span, int ld_kv) {
  WinArgs g = win_args(a, b, t5d_window_head_pad(a.D, a.Dv));
  g.span_off = span.off; g.span_first = span.first; g.ld_kv = ld_kv;
  launch_rows_tiles<true>(s, g);
  T5D_CHECK_LAUNCH("window attention (span)");
  return T5D_OK;
}

int launch_window_wave(hipStream_t s, const t5d_window_attention& a,
                       const t5d_ragged& b, int HP) {
  const WinArgs g = win_args(a, b, HP);
  if (a.dtype == T5D_BF16) launch_wave<bf16_t>(s, g);
  else launch_wave<float>(s, g);
  T5D_CHECK_LAUNCH("window attention (wave)");
  return T5D_OK;
}

}  // namespace t5d

using namespace t5d;

extern "C" int t5d_window_head_pad(int D, int Dv) {
  const int n = D > Dv ? D : Dv;
  if (n <= 0 || n > 1024) return -1;
  for (int p = 32; p <= 256; p *= 2)
    if (n <= p) return p;
  return (n + 63) / 64 * 64;
}

extern "C" int64_t t5d_window_workspace_bytes(int S, int H, int D, int Dv) {
  const int hp = t5d_window_head_pad(D, Dv);
  if (hp < 0 || S <= 0 || H <= 0) return -1;
  return (int64_t)S * H * kMaxSplits * (hp + 2) * 4;
}

extern "C" int t5d_window_attention_run(void* stream, const t5d_window_attention* a,
                                        const t5d_ragged* b, int variant) {
  T5D_REQUIRE(a && b, T5D_EINVAL, "t5d_window_attention_run: null arguments");
  T5D_REQUIRE(a->dtype == T5D_F32 || a->dtype == T5D_BF16, T5D_EINVAL,
              "t5d_window_attention_run: dtype %d", a->dtype);
  T5D_REQUIRE(a->H > 0 && a->G > 0 && a->H % a->G == 0 && a->D > 0 && a->Dv > 0 &&
                  a->window >= 0 && a->H <= 65535 && a->G <= 65535,
              T5D_EINVAL, "t5d_window_attention_run: H=%d G=%d D=%d Dv=%d window=%d",
              a->H, a->G, a->D, a->Dv, a->window);
  T5D_REQUIRE(a->proj && a->key_ring && a->value_ring && a->q_rows && a->out &&
                  b->tok_pos && b->tok_seq && b->seq_off && b->seq_start &&
                  b->seq_slot,
              T5D_EINVAL, "t5d_window_attention_run: null buffer");
  T5D_REQUIRE(b->M > 0 && b->S > 0 && b->S <= 65535 && b->max_len > 0 &&
                  b->max_len <= b->M,
              T5D_EINVAL, "t5d_window_attention_run: M=%d S=%d max_len=%d", b->M,
              b->S, b->max_len);
  T5D_REQUIRE(a->ring > 0 && a->ring % 64 == 0 &&
                  (a->window == 0 || a->ring >= a->window - 1 + b->max_len),
              T5D_EINVAL,
              "t5d_window_attention_run: a ring of %d rows for a window of %d and "
              "portions of %d (multiple of 64, at least window - 1 + portion)",
              a->ring, a->window, b->max_len);
  T5D_REQUIRE(variant >= 0 && variant <= 3, T5D_EINVAL,
              "t5d_window_attention_run: variant %d", variant);
  WinArgs g = win_args(*a, *b, t5d_window_head_pad(a->D, a->Dv));
  T5D_REQUIRE(g.HP > 0, T5D_ELIMIT, "t5d_window_attention_run: head size %d / %d",
              a->D, a->Dv);
  hipStream_t s = as_stream(stream);
  const bool bf16 = a->dtype == T5D_BF16;
  const int GS = step_group(g.gs, g.HP);
  const bool can_step = bf16 && b->max_len == 1 && b->M == b->S && GS > 0;
  const bool can_rows = bf16 && g.HP <= 256 && a->ld_out % 4 == 0;
  T5D_REQUIRE((variant != 1 || can_step) && (variant != 2 || can_rows), T5D_EINVAL,
              "t5d_window_attention_run: variant %d does not cover this call",
              variant);
  if (variant == 1 || (variant == 0 && can_step)) {
    if (g.parts != nullptr) g.splits = step_splits(*a, b->S);
    const dim3 grid(b->S * a->G, g.splits), block(256);
#define T5D_WS(DT_, GS_)                                                     \
  if (g.HP == 32 * DT_ && GS == GS_)                                         \
    hipLaunchKernelGGL((window_step_kernel<DT_, GS_>), grid, block, 0, s, g)
    T5D_WS(1, 1); T5D_WS(1, 2); T5D_WS(1, 4); T5D_WS(1, 8); T5D_WS(1, 16);
    T5D_WS(2, 1); T5D_WS(2, 2); T5D_WS(2, 4); T5D_WS(2, 8); T5D_WS(2, 16);
    T5D_WS(4, 1); T5D_WS(4, 2); T5D_WS(4, 4); T5D_WS(4, 8); T5D_WS(4, 16);
    T5D_WS(8, 1); T5D_WS(8, 2); T5D_WS(8, 4); T5D_WS(8, 8);
#undef T5D_WS
    T5D_CHECK_LAUNCH("window attention (step)");
    if (g.splits > 1) {
      hipLaunchKernelGGL(window_merge_kernel, dim3(b->S * a->H), dim3(64), 0, s, g);
      T5D_CHECK_LAUNCH("window attention (merge)");
    }
    return T5D_OK;
  }
  const int64_t units = (int64_t)b->M * (a->H + 2 * a->G);
  const dim3 agrid((unsigned)((units + 3) / 4)), ablock(256);
  const bool pieces =
      bf16 && g.HP <= 256 &&
      ((a->D | a->Dv | a->off_q | a->off_k | a->off_v | a->ld_proj) & 7) == 0 &&
      (((uintptr_t)a->proj | (uintptr_t)a->q_rows | (uintptr_t)a->key_ring |
        (uintptr_t)a->value_ring | (uintptr_t)a->q_norm | (uintptr_t)a->k_norm) &
       15) == 0;
  if (pieces)
    hipLaunchKernelGGL(window_append_vec_kernel,
                       dim3((unsigned)((units * (g.HP / 8) + 255) / 256)), ablock, 0,
                       s, g);
  else if (bf16)
    hipLaunchKernelGGL(window_append_kernel<bf16_t>, agrid, ablock, 0, s, g);
  else
    hipLaunchKernelGGL(window_append_kernel<float>, agrid, ablock, 0, s, g);
  T5D_CHECK_LAUNCH("window attention (append)");
  // (the rows kernel's loads into LDS want whole 16-byte pieces: rings that start
  // elsewhere go the general way)
  const bool whole = (((uintptr_t)a->key_ring | (uintptr_t)a->value_ring) & 15) == 0;
  if ((variant == 2 || (variant == 0 && can_rows)) && whole) {
    launch_rows_tiles<false>(s, g);
    T5D_CHECK_LAUNCH("window attention (rows)");
    return T5D_OK;
  }
  if (bf16) launch_wave<bf16_t>(s, g);
  else launch_wave<float>(s, g);
  T5D_CHECK_LAUNCH("window attention (wave)");
  return T5D_OK;
}
