"""T5.1.1 encoder forward (t5x/examples/t5/network.py:47-96,182-219,315-343),
run once per batch before the decode loop, on hand-written HIP kernels.

bfloat16: the many-row dense kernel (t5d_gemm_rows: fused residual /
gated-GELU epilogues, value projection written transposed), whole-sequence
self-attention on the matrix cores (t5d_encoder_attention), the embedding
gather and the RMS norm of the decode path.  float32 (the exactness-test
dtype): the float32 dense kernel with the layer norms riding inside it
(t5d_gemm / t5d_norm_gemm) and a vector-ALU attention kernel
(t5d_encoder_attention_f32).  The decode step never calls into this module.
"""

import numpy as np
import torch

from t5x_amd import network


class EncoderKernelWeights:
  """Encoder parameters packed for the HIP kernels (bfloat16 activations)."""

  def __init__(self, cfg, params, device):
    from t5x_amd import ops
    act = torch.bfloat16
    wdt = network._TORCH_DTYPE[cfg.weight_dtype or cfg.dtype]
    enc = params['encoder']
    f = lambda x: network._f32(x, device)
    self.embedding = f(params['token_embedder']['embedding']).to(act).contiguous()
    self.rel_embedding = f(enc['relpos_bias']['rel_embedding']).to(act)
    self.layers = []
    for i in range(cfg.num_encoder_layers):
      p = enc[f'layers_{i}']
      a, m = p['attention'], p['mlp']
      qk = torch.cat([f(a['query']['kernel']), f(a['key']['kernel'])],
                     dim=1).contiguous()
      self.layers.append(dict(
          ln_attn=f(p['pre_attention_layer_norm']['scale']).to(act),
          qk=ops.pack_weight(qk, act, wdt),
          v=ops.pack_weight(f(a['value']['kernel']), act, wdt),
          o=ops.pack_weight(f(a['out']['kernel']), act, wdt),
          ln_mlp=f(p['pre_mlp_layer_norm']['scale']).to(act),
          wi=ops.pack_weight(f(m['wi_0']['kernel']), act, wdt,
                             gate_kernel=f(m['wi_1']['kernel'])),
          wo=ops.pack_weight(f(m['wo']['kernel']), act, wdt)))
    self.ln_final = f(enc['encoder_norm']['scale']).to(act)
    self._bias = {}

  def rel_bias(self, E):
    """[H, 2E-1] bias by (key - query + E - 1), bidirectional buckets."""
    if E not in self._bias:
      bucket = network.relative_position_bucket(np.arange(-(E - 1), E),
                                                bidirectional=True)
      idx = torch.as_tensor(bucket.astype(np.int64),
                            device=self.rel_embedding.device)
      self._bias[E] = self.rel_embedding[:, idx].contiguous()
    return self._bias[E]


def _layers(cfg, w, x, v_t, E, rows, attend):
  """The encoder's layers over x, rows of texts of E positions each or those of an
  EncoderRows; attend(q | k) with the values in v_t.  The norms between layers ride in the
  dense layers on both sides of them, but not with int8 weights, which keep the vector
  units busy (8192 rows of 2048: v 75 us, with the norm inside 83, the gated layer 312 and
  320; a pass of its own takes 15 for the two of them), nor over 32 inputs."""
  from t5x_amd import _lib, ops
  pair = ops.takes_norm(cfg.emb_dim)
  inside = (pair and ops.takes_norm(cfg.num_heads * 64, cfg.mlp_dim) and
            (cfg.weight_dtype or cfg.dtype) == 'bfloat16')

  def residual_and_norm(a, kernel, x, scale):
    if inside:
      return ops.gemm_rows_residual_norm(a, kernel, x, scale)
    x = ops.gemm_rows(a, kernel, residual=x)
    return x, ops.rmsnorm(x, scale)

  def dense(a, kernel):
    return (ops.gemm_rows_of_scaled(a, kernel) if isinstance(a, ops.ScaledRows)
            else ops.gemm_rows(a, kernel))

  xn = ops.rmsnorm(x, w.layers[0]['ln_attn']) if w.layers else None
  for i, l in enumerate(w.layers):
    if pair:
      qk = ops.gemm_rows_pair(xn, l['qk'], l['v'], v_t, E,    # [M, q | k]
                              at=None if rows is None else rows.at)
    else:
      qk = ops.gemm_rows(xn, l['qk'])
      if rows is not None:
        ops.gemm_rows_values(xn, l['v'], rows, out=v_t)
      else:
        ops.gemm_rows(xn, l['v'], out=v_t, layout=_lib.OUT_HEADS_VALUE, E=E,
                      Ep=v_t.shape[2] * 32)
    x, y = residual_and_norm(attend(qk), l['o'], x, l['ln_mlp'])
    h = dense(y, l['wi'])
    if i + 1 < len(w.layers):
      x, xn = residual_and_norm(h, l['wo'], x, w.layers[i + 1]['ln_attn'])
    else:
      x = ops.gemm_rows(h, l['wo'], residual=x)
  return x


def _encode_rows(cfg, w, rows, device):
  """_encode_hip over the rows that there are (ops.EncoderRows)."""
  from t5x_amd import ops
  HD = cfg.num_heads * 64
  bias = w.rel_bias(rows.positions)
  x = ops.embed(w.embedding, rows.ids)
  v_t = torch.zeros((rows.B, cfg.num_heads, (rows.positions + 31) // 32, 64, 32),
                    dtype=x.dtype, device=device)
  def attend(qk):
    return ops.encoder_attention_rows(qk[:, :HD], qk[:, HD:], v_t, bias, rows)

  x = _layers(cfg, w, x, v_t, rows.positions, rows, attend)
  return ops.rmsnorm_rows(x, w.ln_final, rows.row_of).view(rows.B, rows.E,
                                                          cfg.emb_dim)


def _encode_hip(module, params, tokens):
  """bfloat16 encoder on the HIP kernels; tokens [B, E] int64 on the device."""
  from t5x_amd import ops
  cfg, dev = module.config, module._dev()
  key = ('hip', id(params))
  if key not in module._enc_weights:
    module._enc_weights[key] = (params, EncoderKernelWeights(cfg, params, dev))
  w = module._enc_weights[key][1]
  B, E = tokens.shape
  odd = None
  if ops.EncoderRows.covers(B, E) and cfg.emb_dim % 8 == 0:
    rows = ops.EncoderRows(tokens)
    if not rows.odd:
      return _encode_rows(cfg, w, rows, dev)
    odd = True
  if E % 4:
    # The dense kernel's head-layout epilogue takes lengths in multiples of 4:
    # pad with padding tokens (masked keys; their own rows are dropped again).
    tokens = torch.nn.functional.pad(tokens, (0, -E % 4))
    return _encode_positions(cfg, w, tokens, dev, odd)[:, :E].contiguous()
  return _encode_positions(cfg, w, tokens, dev, odd)


def _encode_positions(cfg, w, tokens, dev, odd=None):
  """_encode_hip over every position: padding inside a text is masked by bits.  odd:
  that there is such padding is known (_key_mask)."""
  from t5x_amd import _lib, ops
  B, E = tokens.shape
  H = cfg.num_heads
  HD = H * 64
  lens, bits = _key_mask(tokens, dev, odd)
  Ep = (E + 31) // 32 * 32  # values are stored in blocks of 32 positions
  bias = w.rel_bias(E)
  ids = tokens.reshape(-1).to(torch.int32).contiguous()
  x = ops.embed(w.embedding, ids)
  M = B * E
  v_t = torch.zeros((B, H, Ep // 32, 64, 32), dtype=x.dtype, device=dev)
  def attend(qk):
    return ops.encoder_attention(qk[:, :HD], qk[:, HD:], v_t, bias, lens,
                                 valid_bits=bits)

  x = _layers(cfg, w, x, v_t, E, None, attend)
  return ops.rmsnorm(x, w.ln_final).view(B, E, cfg.emb_dim)


class EncoderKernelWeightsF32:
  """Encoder parameters for the float32 kernels: row-major [K, N] kernels,
  query | key | value fused into one projection."""

  def __init__(self, cfg, params, device):
    from t5x_amd import ops
    f32 = torch.float32
    enc = params['encoder']
    f = lambda x: network._f32(x, device)
    self.embedding = f(params['token_embedder']['embedding']).contiguous()
    self.rel_embedding = f(enc['relpos_bias']['rel_embedding'])
    self.layers = []
    for i in range(cfg.num_encoder_layers):
      p = enc[f'layers_{i}']
      a, m = p['attention'], p['mlp']
      qkv = torch.cat([f(a['query']['kernel']), f(a['key']['kernel']),
                       f(a['value']['kernel'])], dim=1).contiguous()
      self.layers.append(dict(
          ln_attn=f(p['pre_attention_layer_norm']['scale']).contiguous(),
          qkv=ops.pack_weight(qkv, f32),
          o=ops.pack_weight(f(a['out']['kernel']), f32),
          ln_mlp=f(p['pre_mlp_layer_norm']['scale']).contiguous(),
          wi=ops.pack_weight(f(m['wi_0']['kernel']), f32,
                             gate_kernel=f(m['wi_1']['kernel'])),
          wo=ops.pack_weight(f(m['wo']['kernel']), f32)))
    self.ln_final = f(enc['encoder_norm']['scale']).contiguous()
    self._bias = {}

  def rel_bias(self, E):
    """[H, 2E-1] bias by (key - query + E - 1), bidirectional buckets."""
    if E not in self._bias:
      bucket = network.relative_position_bucket(np.arange(-(E - 1), E),
                                                bidirectional=True)
      idx = torch.as_tensor(bucket.astype(np.int64),
                            device=self.rel_embedding.device)
      self._bias[E] = self.rel_embedding[:, idx].contiguous()
    return self._bias[E]


def _key_mask(tokens, dev, odd=None):
  """The padding mask of t5x/examples/t5/network.py:325-328 (token > 0,
  element-wise) as the kernels take it: (lengths, bits).  Padding that is a
  suffix of zeros, the usual case, is a length per row and bits None; a
  padding token inside the text gives the last valid position + 1 and one bit
  per position (ops.token_mask).  odd: take that form at once, instead of waiting
  for the device to say which."""
  from t5x_amd import ops
  B, E = tokens.shape
  if not odd:
    valid = tokens > 0
    lens = valid.sum(dim=1).to(torch.int32)
    prefix = torch.arange(E, device=dev)[None, :] < lens[:, None]
    if bool((prefix == valid).all()):
      return lens.contiguous(), None
  return ops.token_mask(tokens.contiguous())


def _encode_hip_f32(module, params, tokens):
  """float32 encoder on the HIP kernels; tokens [B, E] int64 on the device."""
  from t5x_amd import ops
  cfg, dev = module.config, module._dev()
  key = ('hip_f32', id(params))
  if key not in module._enc_weights:
    module._enc_weights[key] = (params,
                                EncoderKernelWeightsF32(cfg, params, dev))
  w = module._enc_weights[key][1]
  B, E = tokens.shape
  H = cfg.num_heads
  lens, bits = _key_mask(tokens, dev)
  bias = w.rel_bias(E)
  x = ops.embed(w.embedding, tokens.reshape(-1).to(torch.int32).contiguous())
  for l in w.layers:
    qkv = ops.gemm(x, l['qkv'], norm_scale=l['ln_attn'])
    attn = ops.encoder_attention_f32(qkv, bias, lens, H, valid_bits=bits)
    x = ops.gemm(attn, l['o'], residual=x)
    h = ops.gemm(x, l['wi'], norm_scale=l['ln_mlp'])
    x = ops.gemm(h, l['wo'], residual=x)
  return ops.rmsnorm(x, w.ln_final).view(B, E, cfg.emb_dim)


def encode(module, params, encoder_input_tokens):
  """[B, E, emb_dim] of tokens [B, E].  In bfloat16 a text has E rounded up to a
  multiple of 4 positions: tokens do not see the added ones, the padding behind them
  does, whose queries weigh all positions alike (the reference's E, network.py:325-328;
  nothing downstream looks at padding's rows)."""
  cfg, dev = module.config, module._dev()
  tokens = encoder_input_tokens
  if not isinstance(tokens, torch.Tensor):
    tokens = torch.as_tensor(np.asarray(tokens), device=dev)
  tokens = tokens.to(dev).long()
  if cfg.dtype == 'float32':
    return _encode_hip_f32(module, params, tokens)
  if cfg.dtype != 'bfloat16':
    raise ValueError(f'unsupported encoder dtype {cfg.dtype}')
  return _encode_hip(module, params, tokens.contiguous())
