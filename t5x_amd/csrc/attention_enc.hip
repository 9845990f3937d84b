// Encoder self-attention over whole sequences (bfloat16), once per batch:
// out = softmax(Q K^T + relative-position bias + padding mask) V per
// (batch item, head), t5x/examples/t5/layers.py:52-129 with the encoder's
// bidirectional bias (layers.py:560-677) and mask (network.py:325-328).
//
// Two kernels on the matrix cores, chosen by length: enc_attn_short_kernel up to 64
// positions (scores kept in registers between the keys and the values),
// enc_attn_tile_kernel beyond (one pass over the keys, workgroups of 128 queries or 64).
// Both form S^T = K Q^T, keys as matrix rows, so that a lane ends up with 4 consecutive
// keys of ONE query, which is the operand order of out^T = V^T P^T; V is given transposed
// in 32-key blocks ([B, H, Ep / 32, 64, 32], what t5d_gemm_rows' value layout writes).
// Scores are rounded where the reference rounds them.
// Masked keys weigh nothing beside a valid one, and a padded query attends uniformly
// over all keys, as with the reference's -1e10; keys beyond E do not exist.
#include <math.h>

#include "common.h"

namespace t5d {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_e;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_e;

union FragE {
  uint4 u;
  bf16x8_e v;
};

struct EncAttnArgs {
  const bf16_t* q;    // [B*E, q_stride]: head h at columns h*64 .. +64
  const bf16_t* k;    // same layout as q
  const bf16_t* vt;   // [B, H, Ep / 32, 64, 32]: 32-key blocks
  const bf16_t* bias; // [H, 2E-1]: by (key - query + E - 1)
  const int32_t* len; // [B] valid prefix length (with `valid`: last valid + 1)
  const uint32_t* valid;  // optional [B, (E + 31) / 32]: bit e = position e valid
  const int32_t* first;   // ROWS kernels: [B + 1], rows first[b] .. first[b + 1] are
                          // text b's instead of b * E .. (b + 1) * E (t5d_encoder_rows:
                          // every position below len, then one or more of padding)
  const int32_t* order;   // ROWS kernels, optional: [B] the texts, longest first
  bf16_t* out;        // [B*E, H*64]
  int B, H, E, Ep, q_stride, k_stride;
};

// Component 16 dt + 4 g + i of the value vector of position e, from V^T.
__device__ __forceinline__ void value_at(const char* vt, int e, int dt, int gq,
                                         float (&v)[4]) {
  const bf16_t* p = reinterpret_cast<const bf16_t*>(vt) + (size_t)(e >> 5) * 2048 +
                    (16 * dt + 4 * gq) * 32 + (e & 31);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = bf16_to_f32(p[32 * i]);
}

// ---- up to 64 positions: scores kept in registers -------------------------------
// A wavefront's 16 queries against the one block of keys:
//   the scores are formed once and kept as bfloat16 pairs (they ARE bfloat16 values
//   at that point), their maximum and sum with them; then they are turned into P in
//   registers, already in the layout of the matrix cores' B operand: a lane holds
//   keys 4g .. 4g+3 of two neighbouring 16-key tiles, and the V^T operand is read
//   from LDS in that same key order, so P never goes through LDS.
// K and V^T are fetched once per workgroup, 8 KB each, straight from memory into LDS
// (global_load_lds: lane l of an instruction lands at byte 16 l, so the address each
// lane reads from picks the XOR swizzle that makes the operand reads spread over the
// banks); the four wavefronts read their operand fragments from there.
typedef __attribute__((address_space(3))) void* enc_lds_ptr_t;
typedef __attribute__((address_space(1))) const void* enc_glb_ptr_t;

constexpr int kShortEnc = 64;  // its longest text

template <bool ROWS>
__global__ void __launch_bounds__(256)
enc_attn_short_kernel(EncAttnArgs a) {
  __shared__ uint4 s_k[512], s_v[512];
  __shared__ float s_bias[2 * kShortEnc + 16];
  __shared__ uint32_t s_valid[2];
  // what a score is capped by, per key: [0] for a valid query (+inf for a
  // valid key, bf16(-1e10) for a masked one, -inf past E), [1] for a padded
  // query (bf16(-1e10) for every key that exists)
  __shared__ __attribute__((aligned(16))) float s_lim[2][kShortEnc + 16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, gq = lane >> 4;
  const int h = blockIdx.y, b = blockIdx.z;
  const int E = a.E;
  const size_t row0 = ROWS ? a.first[b] : (size_t)b * E;
  const int rows = ROWS ? a.first[b + 1] - a.first[b] : E;  // that are there

  // What this lane fetches of K: chunks (8 keys, 1 KB) wave and wave + 4; lane s
  // lands at slot s & 7 of key s >> 3 and therefore reads piece (s & 7) ^ (s >> 3) of
  // that key (past the end: the last key again).
  const int k_r = lane >> 3, k_piece = (lane & 7) ^ k_r;
  // ... and of V^T (two [64 d][32 keys] blocks, 4 KB each): chunks (16 rows d, 1 KB)
  // wave and wave + 4; lane s lands at slot s & 3 of row s >> 2 and reads piece
  // (s & 3) ^ ((row >> 1) & 1): one swizzle bit, so that the two pieces a lane needs
  // (p and p + 2) stay 32 bytes apart and come with one two-address read, already in
  // operand order.
  const int v_r = lane >> 2, v_piece = (lane & 3) ^ ((v_r >> 1) & 1);
  const char* kbase = reinterpret_cast<const char*>(a.k) + (size_t)h * 128 + k_piece * 16;
  const char* vbase = reinterpret_cast<const char*>(a.vt) +
                      ((size_t)b * a.H + h) * 128 * (size_t)a.Ep;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = wave + 4 * u;
    const int key = min(8 * c + k_r, rows - 1);
    __builtin_amdgcn_global_load_lds(
        (enc_glb_ptr_t)(kbase + (row0 + key) * (size_t)a.k_stride * 2),
        (enc_lds_ptr_t)&s_k[64 * c], 16, 0, 0);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = wave + 4 * u;
    const int blk = min(c >> 2, (a.Ep >> 5) - 1);
    __builtin_amdgcn_global_load_lds(
        (enc_glb_ptr_t)(vbase + (size_t)blk * 4096 + (16 * (c & 3) + v_r) * 64 +
                        v_piece * 16),
        (enc_lds_ptr_t)&s_v[64 * c], 16, 0, 0);
  }

  for (int i = threadIdx.x; i < 2 * E - 1; i += 256)
    s_bias[i] = bf16_to_f32(a.bias[(size_t)h * (2 * E - 1) + i]);
  int n = a.len[b];
  n = n < 0 ? 0 : (n > E ? E : n);
  const int words = (E + 31) >> 5;
  if (threadIdx.x < 2) {
    const int left = n - 32 * threadIdx.x;
    uint32_t prefix = left >= 32 ? 0xffffffffu : (left <= 0 ? 0u : ((1u << left) - 1u));
    if (a.valid && (int)threadIdx.x < words)
      prefix &= a.valid[(size_t)b * words + threadIdx.x];
    s_valid[threadIdx.x] = prefix;
  }
  const int q0 = wave * 16;
  const int qi = min(q0 + l16, rows - 1);
  FragE qb[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
    qb[c].u = *reinterpret_cast<const uint4*>(
        a.q + (row0 + qi) * a.q_stride + h * 64 + 32 * c + 8 * gq);
  __syncthreads();
  const float kMasked = -9999220736.0f;  // bf16(-1e10) exactly, layers.py:309-311
  if (threadIdx.x < kShortEnc + 16) {
    const int i = threadIdx.x;
    const bool ok = i < E && ((s_valid[i >> 5] >> (i & 31)) & 1u) != 0;
    s_lim[0][i] = ok ? INFINITY : (i < E ? kMasked : -INFINITY);
    s_lim[1][i] = i < E ? kMasked : -INFINITY;
  }
  // Key tiles this wavefront walks: the valid prefix when all of its 16 queries are
  // valid (the keys beyond add exact zeros), else every key; none when its queries
  // lie beyond E.
  int my_tiles = 0;
  if (q0 < rows) {
    const bool all_valid =
        q0 + 15 < E && ((s_valid[q0 >> 5] >> (q0 & 31)) & 0xffffu) == 0xffffu;
    my_tiles = ((all_valid ? n : E) + 15) >> 4;
  }
  my_tiles = __builtin_amdgcn_readfirstlane(my_tiles);
  const bool q_valid =
      q0 + l16 < E && ((s_valid[(q0 + l16) >> 5] >> ((q0 + l16) & 31)) & 1u) != 0;
  // All loads have landed; behind the barrier everyone's have.
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // this lane's 4 keys of key tile kt: bias and cap at [16 kt .. 16 kt + 3].
  // Masking is a minimum with the cap: a score never lies below -1e10, so
  // min(x, bf16(-1e10)) is the reference's masked value, min(x, -inf) removes
  // a key that does not exist, min(x, +inf) keeps x.
  const float* bias_g = s_bias + (E - 1) - min(qi, E - 1) + 4 * gq;
  const float* lim_g = s_lim[q_valid ? 0 : 1] + 4 * gq;
  // scores of key tile kt for this lane: keys 16 kt + 4 g + i of query l16
  uint32_t sc[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t) sc[t][0] = sc[t][1] = 0xFF80FF80u;  // -inf
  float m = -3.0e38f, l = 0.f;
  const int swz = l16 & 7;
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) {
    // two key tiles per test: their chains of dependent instructions (LDS read,
    // matrix instruction, rounding, exp) interleave
    if ((kt & ~1) < my_tiles) {
      f32x4_e acc = (f32x4_e){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        FragE kop;
        kop.u = s_k[(16 * kt + l16) * 8 + ((4 * c + gq) ^ swz)];
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop.v, qb[c].v, acc, 0, 0, 0);
      }
      const float4 cap = *reinterpret_cast<const float4*>(lim_g + 16 * kt);
      // two values per rounding instruction; the cap as a median with -inf (one
      // instruction: fminf would first make both operands canonical)
      const uint32_t r01 = pack_bf16x2(acc[0], acc[1]);
      const uint32_t r23 = pack_bf16x2(acc[2], acc[3]);
      const uint32_t x01 = pack_bf16x2(bf16lo_to_f32(r01) + bias_g[16 * kt],
                                       bf16hi_to_f32(r01) + bias_g[16 * kt + 1]);
      const uint32_t x23 = pack_bf16x2(bf16lo_to_f32(r23) + bias_g[16 * kt + 2],
                                       bf16hi_to_f32(r23) + bias_g[16 * kt + 3]);
      float s[4];
      s[0] = __builtin_amdgcn_fmed3f(bf16lo_to_f32(x01), cap.x, -INFINITY);
      s[1] = __builtin_amdgcn_fmed3f(bf16hi_to_f32(x01), cap.y, -INFINITY);
      s[2] = __builtin_amdgcn_fmed3f(bf16lo_to_f32(x23), cap.z, -INFINITY);
      s[3] = __builtin_amdgcn_fmed3f(bf16hi_to_f32(x23), cap.w, -INFINITY);
      const float tm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      const float nm = fmaxf(m, tm);
      float add = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) add += __expf(s[i] - nm);
      l = l * __expf(m - nm) + add;
      m = nm;
      sc[kt][0] = pack_bf16x2(s[0], s[1]);
      sc[kt][1] = pack_bf16x2(s[2], s[3]);
    }
  }
  // combine the 4 lanes (g) that share a query
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {
    const float om = __shfl_xor(m, o, 64), ol = __shfl_xor(l, o, 64);
    const float nm = fmaxf(m, om);
    l = l * __expf(m - nm) + ol * __expf(om - nm);
    m = nm;
  }
  const float inv = 1.0f / l;

  f32x4_e oc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) oc[dt] = (f32x4_e){0.f, 0.f, 0.f, 0.f};
  // V^T operand of a 32-key step: row d = 16 dt + l16, the 8 bytes of keys
  // 4g .. 4g+3 and of keys 16+4g .. 16+4g+3 (pieces g / 2 and 2 + g / 2)
  const int v_swz = (l16 >> 1) & 1;
  const int v_off0 = l16 * 64 + (((gq >> 1) ^ v_swz) * 16) + (gq & 1) * 8;
  auto prob2 = [&](uint32_t packed) {
    return pack_bf16x2(__expf(bf16lo_to_f32(packed) - m) * inv,
                       __expf(bf16hi_to_f32(packed) - m) * inv);
  };
#pragma unroll
  for (int hb = 0; hb < 2; ++hb) {
    FragE pb;
    pb.u.x = prob2(sc[2 * hb][0]);
    pb.u.y = prob2(sc[2 * hb][1]);
    pb.u.z = prob2(sc[2 * hb + 1][0]);
    pb.u.w = prob2(sc[2 * hb + 1][1]);
    const char* blk = reinterpret_cast<const char*>(&s_v[0]) + hb * 4096;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const uint2* vp = reinterpret_cast<const uint2*>(blk + dt * 1024 + v_off0);
      const uint2 lo = vp[0], hi = vp[4];
      FragE va;
      va.u = make_uint4(lo.x, lo.y, hi.x, hi.y);
      oc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va.v, pb.v, oc[dt], 0, 0, 0);
    }
  }
  // A padded query weighs all E positions alike; padding beyond the rows that are there
  // has the values of the padding that is.
  if (ROWS && rows < E && q0 + l16 < rows && !q_valid) {
    const float w = (float)(E - rows) * bf16_to_f32(f32_to_bf16(inv));
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      float v[4];
      value_at(vbase, rows - 1, dt, gq, v);
#pragma unroll
      for (int i = 0; i < 4; ++i) oc[dt][i] = fmaf(w, v[i], oc[dt][i]);
    }
  }
  // oc[dt][i]: out[q = l16][d = 16 dt + 4 g + i]
  if (q0 + l16 < rows) {
    bf16_t* o = a.out + (row0 + q0 + l16) * (size_t)(a.H * 64) + h * 64 + 4 * gq;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      uint2 pk;
      pk.x = pack_bf16x2(oc[dt][0], oc[dt][1]);
      pk.y = pack_bf16x2(oc[dt][2], oc[dt][3]);
      *reinterpret_cast<uint2*>(o + 16 * dt) = pk;
    }
  }
}

// ---- beyond 64 positions: one pass -----------------------------------------------
// A workgroup takes 64 MT queries of one (item, head), a wavefront 16 MT, and walks 64
// keys at a time once: scores as above (rounded where the reference rounds them),
// weights relative to a running maximum that is raised only when a score passes it
// by kMaxSlack powers of two, rounded to bfloat16 as they enter the second product
// and divided by their float32 sum at the end.  K and V^T tiles go from memory
// straight into LDS, one tile ahead in a second pair of buffers, one barrier per
// tile; 16-byte pieces are exchanged within a row (XOR) so that operand reads cover
// all banks.  A masked key is left out (-inf: next to a valid one its weight is an
// exact zero) and a padded query scores 0 with every key that exists (it attends
// uniformly), both in tiles that hold one of the two only; a wavefront of padded
// queries alone forms no scores.
// Which key a matrix row is follows from what the second product wants: rows 4 g + i of
// tiles 2 kb and 2 kb + 1 are keys 8 g + i and 8 g + 4 + i of their 32, so a lane's
// weights are those of 8 keys in a row and V^T comes in one 16-byte read, as it stands.
// (With keys in their order it came in two reads of 8 bytes and 24 moves per tile.)  Of two
// tiles of queries the second holds those 4 further on, so that both share bias entries.
// What bounds it: vector instructions (~260 per tile and wavefront of 32 queries: the
// two roundings of a score, its exponential) against 32 matrix instructions; 49 KB of
// LDS let three workgroups share a CU.  Then how evenly workgroups fall on the CUs: they
// last as long as their text, so where the texts' order is given the longest start first.
// Measured, us, beside the kernels that were here first (up to 512 positions all scores in
// registers as above, two passes beyond) and keys in their order, texts in theirs:
//   7 x 16 heads x 1032 (400 and more valid)   180 -> 71.4
//     rows of 7 x 16 x 1031 (400 and more)            49.5 -> 41.6
//   1 x 12 x 2048                              158 -> 47.1
//   64 x 16 x 512 (all valid)                  261 -> 140 -> 129
//   32 x 12 x 512 (200 and more)              84.6 -> 59.2
//     rows of 32 x 12 x 512 (128 and more)            51.2 -> 41.1 (45.4 without the order)
//   256 x 12 x 66 / 96 / 128 (half and more)  48.1 / 48.7 / 55.3 -> 39.3 / 41.6 / 46.5
//   1 x 12 x 128                               6.6 -> 4.9
// The line to the kernel above lies where its one block of keys ends.  Below, the one
// block needs no running maximum and half or more of a workgroup's queries are not
// there: 512 x 12 x 16 18.2 us above / 30.9 here, 128 x 12 x 40 9.1 / 11.4, 256 x 12 x
// 64 21.8 / 23.5 (with 64 queries per workgroup).
constexpr float kMaxSlack = 8.0f;
constexpr float kLog2eE = 1.4426950408889634f;

template <int MT, bool ROWS>  // 16 queries each per wavefront: 2 or 1
__global__ void __launch_bounds__(256, 3)
enc_attn_tile_kernel(EncAttnArgs a, int tiles) {
  constexpr int KB = 64, QW = 16 * MT;  // keys per tile, queries per wavefront
  __shared__ uint4 s_k0[512], s_v0[512], s_k1[512], s_v1[512];
  // 16 entries before the table (zeros, for queries past the end, which are not stored)
  // and 64 behind it (keys past the end, whose scores are replaced before they are looked
  // at)
  __shared__ float s_bias[16 + 2 * kMaxEncLen + 64];
  __shared__ uint32_t s_valid[kMaxEncLen / 32 + 2];
  // consecutive block ids go round-robin over the 8 XCDs: the tiles of one (item,
  // head) are 8 apart
  const int pair = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / tiles);
  const int at_b = pair / a.H, h = pair - at_b * a.H;
  if (at_b >= a.B) return;
  const int b = ROWS && a.order ? a.order[at_b] : at_b;
  const int tile = (blockIdx.x >> 3) % tiles;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, gq = lane >> 4;
  const int E = a.E;
  const size_t row0 = ROWS ? a.first[b] : (size_t)b * E;
  const int rows = ROWS ? a.first[b + 1] - a.first[b] : E;  // that are there
  if (ROWS && tile * 4 * QW >= rows) return;

  // the pieces this lane fetches: keys (rows of 128 bytes, clamped at the last),
  // V^T (blocks of 32 keys: rows of 64 bytes)
  const char* k_at = reinterpret_cast<const char*>(a.k) + (size_t)h * 128;
  const char* v_at = reinterpret_cast<const char*>(a.vt) +
                     ((size_t)b * a.H + h) * 128 * (size_t)a.Ep;
  int k_row[2], k_piece[2], v_blk[2], v_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int f = (wave * 2 + i) * 64 + lane;
    k_row[i] = f >> 3;
    k_piece[i] = 16 * ((f & 7) ^ (((k_row[i] >> 1) & 1) | ((k_row[i] >> 2) & 6)));
    v_blk[i] = f >> 8;
    const int d = (f >> 2) & 63;
    v_off[i] = d * 64 + 16 * ((f & 3) ^ (3 * ((d >> 3) & 1)));
  }
  const auto fetch = [&](int jt, uint4* sk, uint4* sv) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const size_t row = row0 + min(jt + k_row[i], rows - 1);
      __builtin_amdgcn_global_load_lds(
          (enc_glb_ptr_t)(k_at + row * a.k_stride * 2 + k_piece[i]),
          (enc_lds_ptr_t)(sk + (wave * 2 + i) * 64), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int blk = min((jt >> 5) + v_blk[i], (a.Ep >> 5) - 1);
      __builtin_amdgcn_global_load_lds(
          (enc_glb_ptr_t)(v_at + (size_t)blk * 4096 + v_off[i]),
          (enc_lds_ptr_t)(sv + (wave * 2 + i) * 64), 16, 0, 0);
    }
  };
  fetch(0, s_k0, s_v0);

  int n = a.len[b];
  n = n < 0 ? 0 : (n > E ? E : n);
  // The part of the table that these queries and keys reach (a second tile's queries lie
  // 4 further on), 4 entries per thread requested at a time.
  if (threadIdx.x < 16) s_bias[threadIdx.x] = 0.f;
  {
    const int q_first = tile * 4 * QW;
    const int q_last = min(q_first + 4 * QW, rows) - 1;
    const int lo = max(E - 1 - q_last - 4, 0);
    const int hi = min(E - 1 - q_first + ((ROWS ? n : E) + KB - 1) / KB * KB, 2 * E - 1);
    const bf16_t* table = a.bias + (size_t)h * (2 * E - 1);
    for (int i = lo + threadIdx.x; i < hi; i += 4 * 256) {
      bf16_t v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = table[min(i + 256 * j, hi - 1)];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + 256 * j < hi) s_bias[16 + i + 256 * j] = bf16_to_f32(v[j]);
    }
  }
  const int words = (E + 31) >> 5;
  for (int i = threadIdx.x; i < kMaxEncLen / 32 + 2; i += 256) {
    const int left = n - 32 * i;
    uint32_t prefix =
        left >= 32 ? 0xffffffffu : (left <= 0 ? 0u : ((1u << left) - 1u));
    if (a.valid && i < words) prefix &= a.valid[(size_t)b * words + i];
    s_valid[i] = prefix;
  }
  const int q0 = (tile * 4 + wave) * QW;
  // (of two tiles of queries the second holds those 4 further on)
  const int q_at = MT == 2 ? q0 + 8 * (l16 >> 2) + (l16 & 3) : q0 + l16;
  FragE qb[MT][2];
  int qi[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    qi[mt] = min(q_at + 4 * mt, rows - 1);  // past the end: not stored
#pragma unroll
    for (int c = 0; c < 2; ++c)
      qb[mt][c].u = *reinterpret_cast<const uint4*>(
          a.q + (row0 + qi[mt]) * a.q_stride + h * 64 + 32 * c + 8 * gq);
  }
  __syncthreads();
  // The keys that a padded query weighs here.  Where rows are given, padding is left
  // to the end: one of its rows stands for all of it.
  const int E_here = ROWS ? n : E;
  // Keys each wavefront of the workgroup walks: the valid prefix if all of its
  // queries are valid, else all there are (none past the end).
  int my_keys = 0, wg_keys = 0;
  bool my_valid = false, my_padding = false;  // all queries are
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int qw = (tile * 4 + w) * QW;
    const uint32_t all = MT == 2 ? 0xffffffffu : 0xffffu;
    const uint32_t want =
        qw + QW <= rows ? all : qw < rows ? (1u << (rows - qw)) - 1 : 0;
    const uint32_t there = qw < rows ? (s_valid[qw >> 5] >> (qw & 31)) & want : 0;
    const bool valid = qw < rows && there == want;
    const int keys = qw >= rows ? 0 : valid ? n : E_here;
    if (w == wave) {
      my_keys = keys;
      my_valid = valid;
      my_padding = there == 0;
    }
    wg_keys = max(wg_keys, keys);
  }
  my_keys = __builtin_amdgcn_readfirstlane(my_keys);
  wg_keys = __builtin_amdgcn_readfirstlane(wg_keys);

  bool q_valid[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    q_valid[mt] = (s_valid[qi[mt] >> 5] >> (qi[mt] & 31)) & 1u;
  float mx[MT], l[MT];
  f32x4_e oc[4][MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    mx[mt] = -1e30f;
    l[mt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) oc[dt][mt] = (f32x4_e){0.f, 0.f, 0.f, 0.f};
  }
  const int k_read = (8 * (l16 >> 2) + (l16 & 3)) * 8, k_x = l16 >> 1;
  const int v_read = l16 * 4 + (gq ^ (3 * (l16 >> 3)));
  const auto attend = [&](int jt, const uint4* sk, const uint4* sv) {
    if (jt >= my_keys) return;
    FragE pb[2][MT];
    if (my_padding) {
      // every key that exists weighs the same: no scores
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = jt + 32 * kb + 8 * gq + 2 * e;
          w[e] = (key < E_here ? 0x3F80u : 0u) | (key + 1 < E_here ? 0x3F800000u : 0u);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            l[mt] += (float)((key < E_here) + (key + 1 < E_here));
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          pb[kb][mt].u = make_uint4(w[0], w[1], w[2], w[3]);
      }
    } else {
    f32x4_e s[4][MT];
    FragE kf[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        kf[t][c].u = sk[(32 * (t >> 1) + 4 * (t & 1)) * 8 + k_read + ((4 * c + gq) ^ k_x)];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) s[t][mt] = (f32x4_e){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          s[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][c].v, qb[mt][c].v,
                                                             s[t][mt], 0, 0, 0);
    // bias by key - query: 4 keys further on is 4 queries further back
    const float* near = s_bias + 16 + (E - 1) - min(qi[0], E - 1) + jt + 8 * gq;
    float bias[2][MT + 1][4];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j <= MT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          bias[kb][j][i] = near[32 * kb + 4 * (j - (MT - 1)) + i];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float* add = bias[t >> 1][(t & 1) - mt + MT - 1];
        const uint32_t r01 = pack_bf16x2(s[t][mt][0], s[t][mt][1]);
        const uint32_t r23 = pack_bf16x2(s[t][mt][2], s[t][mt][3]);
        const uint32_t x01 =
            pack_bf16x2(bf16lo_to_f32(r01) + add[0], bf16hi_to_f32(r01) + add[1]);
        const uint32_t x23 =
            pack_bf16x2(bf16lo_to_f32(r23) + add[2], bf16hi_to_f32(r23) + add[3]);
        s[t][mt][0] = bf16lo_to_f32(x01);
        s[t][mt][1] = bf16hi_to_f32(x01);
        s[t][mt][2] = bf16lo_to_f32(x23);
        s[t][mt][3] = bf16hi_to_f32(x23);
      }
    const uint32_t v0 = s_valid[jt >> 5], v1 = s_valid[(jt >> 5) + 1];
    if (!my_valid) {  // a padded query scores 0
      asm volatile("");  // (a branch: the compiler would select in every tile)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[t][mt][i] = q_valid[mt] ? s[t][mt][i] : 0.f;
    }
    if ((v0 & v1) != 0xffffffffu) {  // with keys that it does weigh, if they exist
      asm volatile("");
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = 32 * (t >> 1) + 8 * gq + 4 * (t & 1) + i;
          const bool exists = jt + key < E_here;
          // (of given rows the keys below E_here are the valid ones)
          const bool ok = ROWS ? exists : ((t < 2 ? v0 : v1) >> (key & 31)) & 1u;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            s[t][mt][i] = (q_valid[mt] ? ok : exists) ? s[t][mt][i] : -INFINITY;
        }
    }
    bool raise = false;
    float top[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      top[mt] = -INFINITY;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) top[mt] = fmaxf(top[mt], s[t][mt][i]);
      top[mt] = rows_max(top[mt]) * kLog2eE;
      raise |= top[mt] > mx[mt] + kMaxSlack;
    }
    if (__builtin_amdgcn_ballot_w64(raise) != 0) {
      asm volatile("");
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        // (of those queries alone whose own score asks for it: what a query gets does
        // not depend on the ones beside it)
        const float to = top[mt] > mx[mt] + kMaxSlack ? top[mt] : mx[mt];
        const float alpha = __builtin_amdgcn_exp2f(mx[mt] - to);
        mx[mt] = to;
        l[mt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
          for (int i = 0; i < 4; ++i) oc[dt][mt][i] *= alpha;
          asm volatile("" : "+v"(oc[dt][mt]));
        }
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[t][mt][i], kLog2eE, -mx[mt]));
          s[t][mt][i] = p;
          sum += p;
        }
      l[mt] += sum;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        pb[kb][mt].u = make_uint4(pack_bf16x2(s[2 * kb][mt][0], s[2 * kb][mt][1]),
                                  pack_bf16x2(s[2 * kb][mt][2], s[2 * kb][mt][3]),
                                  pack_bf16x2(s[2 * kb + 1][mt][0], s[2 * kb + 1][mt][1]),
                                  pack_bf16x2(s[2 * kb + 1][mt][2], s[2 * kb + 1][mt][3]));
    }
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      FragE va[4];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        va[dt].u = sv[kb * 256 + dt * 64 + v_read];
      }
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          oc[dt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              va[dt].v, pb[kb][mt].v, oc[dt][mt], 0, 0, 0);
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
  // (every tile that is fetched is met before the end.  wg_keys >= 1, as a workgroup has a
  // query, which is valid or walks all keys; but not of given rows, where a text may have
  // no token: the first tile has been fetched all the same)
  for (int jt = 0; (ROWS && jt == 0) || jt < wg_keys; jt += 2 * KB) {
    meet();
    if (jt + KB < wg_keys) fetch(jt + KB, s_k1, s_v1);
    attend(jt, s_k0, s_v0);
    if (jt + KB >= wg_keys) break;
    meet();
    if (jt + 2 * KB < wg_keys) fetch(jt + 2 * KB, s_k0, s_v0);
    attend(jt + KB, s_k1, s_v1);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    float sum = rows_sum(l[mt]);
    const int q = q_at + 4 * mt;
    if (q >= rows) continue;
    // (such a query's maximum is 0, or was never raised: its keys weigh 1)
    if (ROWS && n < E && q >= n) {
      const float w = (float)(E - n);
      sum += w;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        float v[4];
        value_at(v_at, n, dt, gq, v);
#pragma unroll
        for (int i = 0; i < 4; ++i) oc[dt][mt][i] = fmaf(w, v[i], oc[dt][mt][i]);
      }
    }
    const float inv = 1.0f / sum;
    bf16_t* o = a.out + (row0 + q) * (size_t)(a.H * 64) + h * 64 + 4 * gq;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      *reinterpret_cast<uint2*>(o + 16 * dt) =
          make_uint2(pack_bf16x2(oc[dt][mt][0] * inv, oc[dt][mt][1] * inv),
                     pack_bf16x2(oc[dt][mt][2] * inv, oc[dt][mt][3] * inv));
  }
}

// ---- float32 -------------------------------------------------------------------
// The exactness-test dtype: plain vector arithmetic, one wavefront per query
// row.  Scores (lane = key, ascending head dim), bias and mask summed first and
// added to the score as the reference does (a masked pair ends at exactly
// -1e10, so a padded query attends uniformly), softmax over all E keys, then
// lane = head dim accumulates the normalised weights times V in ascending key
// order.  qkv rows hold q | k | v (H*64 columns each).
struct EncAttnF32Args {
  const float* qkv;   // [B*E, 3*H*64]
  const float* bias;  // [H, 2E-1], by (key - query + E - 1)
  const int32_t* len; // [B]
  const uint32_t* valid;  // optional [B, (E + 31) / 32], as EncAttnArgs
  float* out;         // [B*E, H*64]
  int H, E;
};

constexpr int kEncF32Rows = 4;  // query rows (wavefronts) per workgroup
constexpr int kHeadDim = 64;

__global__ void __launch_bounds__(64 * kEncF32Rows)
enc_attn_f32_kernel(EncAttnF32Args a) {
  __shared__ float s_w[kEncF32Rows][kMaxEncLen];
  __shared__ __attribute__((aligned(16))) float s_q[kEncF32Rows][kHeadDim];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = blockIdx.x * kEncF32Rows + wave;
  const int h = blockIdx.y, b = blockIdx.z;
  if (e >= a.E) return;  // whole wavefronts; no workgroup barrier below
  const int HD = a.H * kHeadDim, row_stride = 3 * HD;
  const int n = min(max(a.len[b], 0), a.E);
  const float* base = a.qkv + (size_t)b * a.E * row_stride + h * kHeadDim;
  s_q[wave][lane] = base[(size_t)e * row_stride + lane];
  const float* bias = a.bias + (size_t)h * (2 * a.E - 1) + (a.E - 1) - e;
  const int words = (a.E + 31) >> 5;
  auto is_valid = [&](int pos) {
    return pos < n &&
           (a.valid == nullptr ||
            ((a.valid[(size_t)b * words + (pos >> 5)] >> (pos & 31)) & 1u) != 0);
  };
  const bool q_valid = is_valid(e);

  float m = -INFINITY;
  for (int j = lane; j < a.E; j += 64) {
    const float4* kr =
        reinterpret_cast<const float4*>(base + (size_t)j * row_stride + HD);
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < kHeadDim / 4; ++c) {
      const float4 kv = kr[c];
      const float4 qv = *reinterpret_cast<const float4*>(&s_q[wave][4 * c]);
      s = fmaf(qv.x, kv.x, s);
      s = fmaf(qv.y, kv.y, s);
      s = fmaf(qv.z, kv.z, s);
      s = fmaf(qv.w, kv.w, s);
    }
    const float mask = (q_valid && is_valid(j)) ? 0.f : -1e10f;
    const float x = s + (mask + bias[j]);
    s_w[wave][j] = x;
    m = fmaxf(m, x);
  }
  m = wave_max(m);
  float sum = 0.f;
  for (int j = lane; j < a.E; j += 64) {
    const float p = expf(s_w[wave][j] - m);
    s_w[wave][j] = p;
    sum += p;
  }
  sum = wave_sum(sum);
  // s_w[wave] is written and read by this wavefront only
  float acc = 0.f;
  const float* vr = base + 2 * HD + lane;
  for (int j = 0; j < a.E; ++j)
    acc = fmaf(s_w[wave][j] / sum, vr[(size_t)j * row_stride], acc);
  a.out[((size_t)b * a.E + e) * HD + h * kHeadDim + lane] = acc;
}

// Whether enc_attn_tile_kernel takes 64 queries per workgroup: while those are at most
// 4 per CU (3 run at a time).  A workgroup of 128 lasts longer than one of 64, whatever
// else the chip does, and longer still if some of its queries are padding (they then
// walk all keys beside the others'): one text of 500 tokens had been faster two passes
// and 64 queries at a time.  Measured, us with 128 / 64 (workgroups of 64):
//   1 x 12 heads x 512, 300 and more valid (96)   17.9 / 13.4
//   2 x 12 x 512, 128 and more (192)              18.7 / 13.6
//   8 x 12 x 200, 80 and more (384)               10.6 / 10.7
//   8 x 12 x 512, 200 and more (768)              26.9 / 21.6
//   4 x 16 x 1032, 400 and more (1088)            53.4 / 49.7
//   16 x 12 x 512, 200 and more (1536)            37.8 / 36.9
//   32 x 12 x 200, 80 and more (1536)             20.0 / 22.6
//   7 x 16 x 1032, 400 and more (1904)            71.5 / 73.8
// Over given rows (there are `rows` of them) as many workgroups count as hold some, and
// padding is one row of a text: 64 pay up to more of them, and longer where texts are long
// (128 / 64, workgroups of 64):
//   3 x 16 heads x 1031, 257 and more (480)       27.9 / 20.5
//   17 x 12 x 512, 128 and more (1176)            28.4 / 26.3
//   7 x 16 x 1031, 400 and more (1296)            45.5 / 41.6
//   10 x 16 x 1500, 375 and more (2032)           72.9 / 69.5
//   31 x 12 x 512, 128 and more (2064)            39.5 / 41.8
//   15 x 16 x 1031, 257 and more (2560)           68.7 / 72.4
//   70 x 12 x 128, 32 and more (1404)             16.7 / 18.1
//   45 x 12 x 200, 50 and more (1152)             19.3 / 21.0
//   45 x 16 x 200, 50 and more (1536)             22.5 / 26.9
static bool one_pass_64(int B, int H, int E, int rows) {
  if (rows > 0)
    return (int64_t)H * (rows / 64 + B / 2) <= (rows >= (int64_t)B * 192 ? 1800 : 1000);
  return (int64_t)B * H * ((E + 63) / 64) <= 1024;
}

}  // namespace t5d

using namespace t5d;

extern "C" int t5d_encoder_attention(void* stream, const void* q, const void* k,
                                     const void* v_t, const void* rel_bias,
                                     const int32_t* enc_len,
                                     const uint32_t* valid_bits, void* out,
                                     int B, int H, int E, int Ep, int q_stride,
                                     int k_stride) {
  return t5d_encoder_attention_variant(stream, q, k, v_t, rel_bias, enc_len,
                                       valid_bits, out, B, H, E, Ep, q_stride,
                                       k_stride, 0);
}

static int encoder_attention(void* stream, const void* q, const void* k, const void* v_t,
                             const void* rel_bias, const int32_t* enc_len,
                             const uint32_t* valid_bits, const int32_t* first,
                             const int32_t* order, int rows, int most, void* out,
                             int B, int H, int E, int Ep, int q_stride, int k_stride) {
  T5D_REQUIRE(q && k && v_t && rel_bias && enc_len && out, T5D_EINVAL,
              "t5d_encoder_attention: null pointer");
  T5D_REQUIRE(B > 0 && H > 0 && E > 0 && Ep >= E && Ep % 32 == 0,
              T5D_EINVAL, "t5d_encoder_attention: B=%d H=%d E=%d Ep=%d", B, H,
              E, Ep);
  T5D_REQUIRE(q_stride >= H * 64 && k_stride >= H * 64 && q_stride % 8 == 0 &&
                  k_stride % 8 == 0,
              T5D_EINVAL, "t5d_encoder_attention: row strides %d / %d", q_stride,
              k_stride);
  T5D_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 &&
                  ((uintptr_t)v_t % 16) == 0 && ((uintptr_t)out % 8) == 0,
              T5D_EINVAL, "t5d_encoder_attention: operand alignment");
  T5D_REQUIRE(E <= kMaxEncLen, T5D_ELIMIT,
              "t5d_encoder_attention: E=%d beyond %d", E, kMaxEncLen);
  T5D_REQUIRE(H <= 65535 && B <= 65535 &&
                  (E <= kShortEnc ||  // (one dimension: fewer than 2^32 threads)
                   ((int64_t)B * H + 7) / 8 * 8 * ((E + 127) / 128) < (1LL << 24)),
              T5D_ELIMIT, "t5d_encoder_attention: H=%d B=%d beyond the launch grid",
              H, B);
  EncAttnArgs a;
  a.q = (const bf16_t*)q; a.k = (const bf16_t*)k; a.vt = (const bf16_t*)v_t;
  a.bias = (const bf16_t*)rel_bias; a.len = enc_len; a.out = (bf16_t*)out;
  a.valid = valid_bits; a.first = first; a.order = order;
  a.B = B; a.H = H; a.E = E; a.Ep = Ep; a.q_stride = q_stride; a.k_stride = k_stride;
  if (E <= kShortEnc) {
    if (first)
      hipLaunchKernelGGL(enc_attn_short_kernel<true>, dim3(1, H, B), dim3(256), 0,
                         as_stream(stream), a);
    else
      hipLaunchKernelGGL(enc_attn_short_kernel<false>, dim3(1, H, B), dim3(256), 0,
                         as_stream(stream), a);
  } else {
    const bool low = one_pass_64(B, H, most, rows);
    const int tiles = low ? (most + 63) / 64 : (most + 127) / 128;
    const dim3 groups(((unsigned)B * H + 7) / 8 * 8 * tiles);
#define T5D_ENC(MT_, ROWS_)                                                       \
  hipLaunchKernelGGL((enc_attn_tile_kernel<MT_, ROWS_>), groups, dim3(256), 0,    \
                     as_stream(stream), a, tiles)
    if (low && first) T5D_ENC(1, true);
    else if (low) T5D_ENC(1, false);
    else if (first) T5D_ENC(2, true);
    else T5D_ENC(2, false);
#undef T5D_ENC
  }
  T5D_CHECK_LAUNCH("t5d_encoder_attention");
  return T5D_OK;
}

extern "C" int t5d_encoder_attention_variant(
    void* stream, const void* q, const void* k, const void* v_t,
    const void* rel_bias, const int32_t* enc_len, const uint32_t* valid_bits,
    void* out, int B, int H, int E, int Ep, int q_stride, int k_stride,
    int variant) {
  T5D_REQUIRE(variant >= 0 && variant <= 2 && (variant != 2 || E <= 512),
              T5D_EINVAL,
              "t5d_encoder_attention_variant: variant %d (0, 1, and 2 where "
              "E <= 512)",
              variant);
  return encoder_attention(stream, q, k, v_t, rel_bias, enc_len, valid_bits, nullptr,
                           nullptr, 0, E, out, B, H, E, Ep, q_stride, k_stride);
}

extern "C" int t5d_encoder_attention_rows(
    void* stream, const void* q, const void* k, const void* v_t, const void* rel_bias,
    const int32_t* enc_len, const int32_t* first, int most, void* out, int B, int H,
    int E, int Ep, int q_stride, int k_stride) {
  return t5d_encoder_attention_ordered(stream, q, k, v_t, rel_bias, enc_len, first,
                                       nullptr, 0, most, out, B, H, E, Ep, q_stride,
                                       k_stride);
}

extern "C" int t5d_encoder_attention_ordered(
    void* stream, const void* q, const void* k, const void* v_t, const void* rel_bias,
    const int32_t* enc_len, const int32_t* first, const int32_t* order, int rows,
    int most, void* out, int B, int H, int E, int Ep, int q_stride, int k_stride) {
  T5D_REQUIRE(first && most > 0 && most <= (E + 3) / 4 * 4 && rows >= 0, T5D_EINVAL,
              "t5d_encoder_attention_ordered: first %p, %d rows, at most %d of a text of %d",
              (const void*)first, rows, most, E);
  return encoder_attention(stream, q, k, v_t, rel_bias, enc_len, nullptr, first, order,
                           rows, most, out, B, H, E, Ep, q_stride, k_stride);
}

extern "C" int t5d_encoder_attention_f32(void* stream, const float* qkv,
                                         const float* rel_bias,
                                         const int32_t* enc_len,
                                         const uint32_t* valid_bits,
                                         float* out, int B, int H, int E) {
  T5D_REQUIRE(qkv && rel_bias && enc_len && out, T5D_EINVAL,
              "t5d_encoder_attention_f32: null pointer");
  T5D_REQUIRE(B > 0 && H > 0 && E > 0, T5D_EINVAL,
              "t5d_encoder_attention_f32: B=%d H=%d E=%d", B, H, E);
  T5D_REQUIRE(E <= kMaxEncLen, T5D_ELIMIT,
              "t5d_encoder_attention_f32: E=%d beyond %d", E, kMaxEncLen);
  T5D_REQUIRE(H <= 65535 && B <= 65535, T5D_ELIMIT,
              "t5d_encoder_attention_f32: H=%d B=%d beyond the launch grid", H,
              B);
  T5D_REQUIRE(((uintptr_t)qkv % 16) == 0, T5D_EINVAL,
              "t5d_encoder_attention_f32: qkv must be 16-byte aligned");
  EncAttnF32Args a;
  a.qkv = qkv; a.bias = rel_bias; a.len = enc_len; a.out = out;
  a.valid = valid_bits;
  a.H = H; a.E = E;
  dim3 grid((E + kEncF32Rows - 1) / kEncF32Rows, H, B);
  hipLaunchKernelGGL(enc_attn_f32_kernel, grid, dim3(64 * kEncF32Rows), 0,
                     as_stream(stream), a);
  T5D_CHECK_LAUNCH("t5d_encoder_attention_f32");
  return T5D_OK;
}
