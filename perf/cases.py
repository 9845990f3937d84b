"""The work this framework is used for, as cases that can be timed and compared.

T5.1.1 encoder-decoder models: whole predictions (encoder, cross keys / values,
beam search or sampling as replayed graphs) and the encoder alone.  Decoder-only
models, of the hybrid family (windowed attention, two kinds of linear
recurrences) and of the latent family (latent attention, hyper-connections,
experts by token table): prompts fed to the cache, single steps of many requests
or of one, and whole generations.

Weights are random, with the shapes of the models that bench.py measures.  Where
tokens are chosen, the output layer holds a successor for every token that stands
out of the others by about the margin it has in a trained model, so a choice does
not hang on the last bit of a logit.

`exact` restates the models in float64 (parallel over positions: chosen tokens are
found as the fixed point of one forward over the whole sequence).
"""

import functools
import math

import numpy as np
import torch

from t5x_amd import decoding
from t5x_amd import hybrid
from t5x_amd import models
from t5x_amd import network

VOCAB = 32128
EPS = 1e-6
DEV = 'cuda'

# T5.1.1 sizes: width, heads (of 64), feed-forward, layers of each stack
T5 = {'small': (512, 6, 1024, 8), 'base': (768, 12, 2048, 12),
      'large': (1024, 16, 2816, 24), 'xl': (2048, 32, 5120, 24)}
# decoder-only sizes: width -> feed-forward; 8 layers, heads of 128
FF = {768: 2048, 1024: 2816, 2048: 5120}
LAYERS, HEAD, WINDOW, LOW = 8, 128, 1024, 64
RANK, STREAMS, EXPERTS, TOP = 512, 4, 64, 4


def listed():
  return [
      # The smallest whole call: a few short texts, greedy, in float32 (the dtype
      # of exactness tests and of users without bfloat16 checkpoints).
      dict(name='predict-small-f32', kind='predict', size='small', dtype='float32',
           batch=8, beams=0, temperature=0.0, topk=0, enc=64, enc_min=64,
           length=32),
      # The headline workload: beam search of T5.1.1-base over documents of
      # 128..512 tokens.
      dict(name='predict-base-beam4', kind='predict', size='base',
           dtype='bfloat16', batch=32, beams=4, temperature=0.0, topk=0, enc=512,
           enc_min=128, length=128),
      # Sampling from a larger model: one row per text, top-k with noise.
      dict(name='predict-large-sample', kind='predict', size='large',
           dtype='bfloat16', batch=64, beams=0, temperature=0.7, topk=40, enc=512,
           enc_min=512, length=128),
      # Weight-only int8, the way a model of this size is served on one GPU.
      dict(name='predict-xl-int8-beam4', kind='predict', size='xl', dtype='int8',
           batch=16, beams=4, temperature=0.0, topk=0, enc=512, enc_min=512,
           length=64),
      # The encoder on its own (embeddings for retrieval, scoring, the stage in
      # front of every decode): a full batch of texts up to 512 tokens ...
      dict(name='encode-base', kind='encode', size='base', batch=32, enc=512,
           enc_min=128),
      # ... and few long ones of a length that no tile divides.
      dict(name='encode-large-long', kind='encode', size='large', batch=7,
           enc=1031, enc_min=400),
      # Long prompts into the cache of a hybrid model.
      dict(name='prefill-hybrid', kind='prefill', family='hybrid', width=1024,
           batch=4, longest=4096, shortest=4096),
      # Prompts of chat length, every one its own, of the same model.
      dict(name='prefill-hybrid-ragged', kind='prefill', family='hybrid',
           width=1024, batch=40, longest=611, shortest=3),
      # One request being answered: a step of a single row, all latency.
      dict(name='step-hybrid-1', kind='step', family='hybrid', width=1024, rows=1,
           position=2047),
      # The whole of a generation request batch: prefill, then replayed steps.
      dict(name='generate-hybrid', kind='generate', family='hybrid', width=1024,
           batch=64, longest=300, shortest=40, new=64),
      # Long prompts into the cache of a latent model.
      dict(name='prefill-latent', kind='prefill', family='latent', width=1024,
           batch=4, longest=4096, shortest=4096),
      # A serving step of a latent model: 64 requests, one token each.
      dict(name='step-latent-64', kind='step', family='latent', width=1024,
           rows=64, position=4100),
  ]


def _log(rng, lo, hi):
  """A whole number between lo and hi, spread over its logarithm."""
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  kind = rng.choice(['predict', 'encode', 'prefill', 'prefill', 'step', 'generate'])
  family = rng.choice(['hybrid', 'latent'])
  width = rng.choice([768, 1024, 1024, 2048])
  if kind == 'predict':
    size, dtype, loop = rng.choice([
        ('small', 'float32', 'greedy'), ('small', 'bfloat16', 'beam'),
        ('base', 'bfloat16', 'beam'), ('base', 'bfloat16', 'greedy'),
        ('large', 'bfloat16', 'sample'), ('large', 'int8', 'beam')])
    beams = rng.choice([2, 3, 4, 5]) if loop == 'beam' else 0
    rows = _log(rng, 1, 16 if dtype == 'float32' else 64)
    enc = _log(rng, 20, 512)
    return dict(kind=kind, size=size, dtype=dtype, beams=beams,
                batch=max(1, rows // max(1, beams)),
                temperature=0.7 if loop == 'sample' else 0.0,
                topk=40 if loop == 'sample' else 0, enc=enc,
                enc_min=rng.randint(max(1, enc // 4), enc),
                length=_log(rng, 8, 32 if dtype == 'float32' else 96))
  if kind == 'encode':
    size = rng.choice(['small', 'base', 'large'])
    enc = _log(rng, 17, 1500)
    return dict(kind=kind, size=size, batch=max(1, _log(rng, 200, 16384) // enc),
                enc=enc, enc_min=rng.randint(max(1, enc // 4), enc))
  if kind == 'prefill':
    longest = _log(rng, 25, 4096)
    return dict(kind=kind, family=family, width=width,
                batch=max(1, min(64, _log(rng, 100, 16384) // longest)),
                longest=longest,
                shortest=rng.choice([longest, rng.randint(1, longest)]))
  if kind == 'step':
    return dict(kind=kind, family=family, width=width, rows=_log(rng, 1, 64),
                position=_log(rng, 40, 4300))
  longest = _log(rng, 8, 600)
  return dict(kind=kind, family=family, width=width, batch=_log(rng, 1, 64),
              longest=longest, shortest=rng.randint(1, longest),
              new=_log(rng, 8, 64))


# ------------------------------------------------------------------------------
# Parameters: random weights whose bfloat16 image is what the model computes with
# ------------------------------------------------------------------------------


class _Random:
  """Tensors from one generator, on the device."""

  def __init__(self, seed, bf16):
    self.gen = torch.Generator(device=DEV)
    self.gen.manual_seed(seed)
    self.bf16 = bf16

  def normal(self, *shape):
    return torch.randn(shape, generator=self.gen, device=DEV)

  def round(self, t):
    return t.to(torch.bfloat16).float() if self.bf16 else t

  def linear(self, k, n, scale=None):
    """[k, n] with k inputs."""
    return self.round(self.normal(k, n) * (scale or k ** -0.5))


def _successors(seed=7):
  """What follows each token: one cycle over all tokens but 0 (padding) and 1
  (end of text)."""
  order = np.random.RandomState(seed).permutation(VOCAB - 2) + 2
  after = np.zeros(VOCAB, np.int64)
  after[order] = np.roll(order, -1)
  return after


def _head(r, embedding, gain):
  """[width, VOCAB] output layer: random, each column leaning `gain` towards the
  embedding of the token it succeeds; nothing speaks for tokens 0 and 1."""
  d = embedding.shape[1]
  lean = torch.zeros_like(embedding)
  after = torch.as_tensor(_successors(), device=DEV)
  lean[after[2:]] = embedding[2:]
  w = (r.normal(VOCAB, d) + gain * lean) * d ** -0.5
  w[:2] = 0
  return r.round(w.t().contiguous())


# How far the successor stands out: it has a share of 0.95 and more on average.
T5_GAIN = {'small': 0.75, 'base': 0.65, 'large': 0.7, 'xl': 0.42}
HYBRID_GAIN = {768: 0.75, 1024: 0.65, 2048: 0.47}
LATENT_GAIN = {768: 0.6, 1024: 0.52, 2048: 0.4}


def _t5_params(case):
  d, H, F, layers = T5[case['size']]
  r = _Random(11, case.get('dtype') != 'float32')
  hd = H * 64
  norm = lambda: {'scale': r.round(1.0 + 0.1 * r.normal(d))}
  lin = lambda k, n, s=None: {'kernel': r.linear(k, n, s)}
  attn = lambda: {'query': lin(d, hd, (64 * d) ** -0.5), 'key': lin(d, hd),
                  'value': lin(d, hd), 'out': lin(hd, d, (2 * layers * hd) ** -0.5)}
  mlp = lambda: {'wi_0': lin(d, F), 'wi_1': lin(d, F),
                 'wo': lin(F, d, (2 * layers * F) ** -0.5)}
  rel = lambda: {'rel_embedding': r.linear(H, 32, 0.5)}
  embedding = r.round(r.normal(VOCAB, d))
  enc = {'relpos_bias': rel(), 'encoder_norm': norm()}
  dec = {'relpos_bias': rel(), 'decoder_norm': norm(),
         'logits_dense': {'kernel': _head(r, embedding, T5_GAIN[case['size']])}}
  for i in range(layers):
    enc[f'layers_{i}'] = {'pre_attention_layer_norm': norm(), 'attention': attn(),
                          'pre_mlp_layer_norm': norm(), 'mlp': mlp()}
    dec[f'layers_{i}'] = {
        'pre_self_attention_layer_norm': norm(), 'self_attention': attn(),
        'pre_cross_attention_layer_norm': norm(),
        'encoder_decoder_attention': attn(), 'pre_mlp_layer_norm': norm(),
        'mlp': mlp()}
  return {'token_embedder': {'embedding': embedding}, 'encoder': enc,
          'decoder': dec}


def _lm_config(case):
  """config.json of a decoder-only model: two thirds recurrent layers and a
  quarter windowed attention, or latent attention with shared latents and
  mixtures behind a dense first feed-forward."""
  W, F = case['width'], FF[case['width']]
  H = W // HEAD
  size = {'heads': H, 'dim': HEAD, 'vdim': HEAD}
  window = {'mask': {'size': WINDOW}, 'scale': HEAD ** -0.5}
  if case['family'] == 'hybrid':
    mixers = {'channel_delta': {**size, 'kv_heads': H, 'conv': 4},
              'gla': {**size, 'tau': 12.0},
              'attention': {**size, **window, 'kv_heads': max(1, H // 4)}}
    order = ['channel_delta', 'gla', 'channel_delta', 'attention'] * 2
    return {'architecture': 'Mokivik', 'width': W, 'vocab': VOCAB,
            'norm': {'eps': EPS},
            'layers': [{'type': t, 'mixer': mixers[t],
                        'mlp': {'kind': 'dense', 'ff': F, 'limit': 7.0}}
                       for t in order]}
  mixer = {**size, **window, 'q_rank': W // 2, 'kv_rank': RANK}
  moe = {'kind': 'moe', 'router': {'experts': EXPERTS, 'top': TOP},
         'expert': {'ff': F // 8, 'limit': 7.0},
         'shared': {'ff': F // 2, 'limit': 7.0}}
  layers = [{'type': 'latent_attention',
             'mixer': dict(mixer, kv_from=i // 4 * 4 + 1) if i % 4 > 1 else mixer,
             'mlp': moe if i else {'kind': 'dense', 'ff': F}}
            for i in range(LAYERS)]
  return {'architecture': 'Nutizen', 'width': W, 'vocab': VOCAB,
          'norm': {'eps': EPS}, 'embedding': {'scale': 1.0}, 'streams': STREAMS,
          'layers': layers}


def _lm_params(case, config):
  """Parameters by tensor name, linear weights [out, in]."""
  W, r = config['width'], _Random(13, True)
  out = {}

  # branches that are not normed behind add up: they start out small
  small = (2 * LAYERS) ** -0.5 if case['family'] == 'latent' else 1.0

  def linear(name, n, k, factor=1.0):
    out[name] = r.linear(n, k, factor * k ** -0.5)

  def unit(prefix, F):
    linear(prefix + 'gate', F, W)
    linear(prefix + 'up', F, W)
    linear(prefix + 'down', W, F, small)

  norm = lambda n: 1.0 + 0.1 * r.normal(n)
  out['embed'] = r.round(r.normal(VOCAB, W))
  gain = (HYBRID_GAIN if case['family'] == 'hybrid' else LATENT_GAIN)[W]
  if case['kind'] != 'generate':
    gain = 0.0
  out['head'] = _head(r, out['embed'], gain).t().contiguous()
  out['final.norm'] = norm(W)
  for i, layer in enumerate(config['layers']):
    m, mlp, p = layer['mixer'], layer['mlp'], f'l{i}.'
    kind, q = layer['type'], p + 'mix.'
    H, D, Dv = m['heads'], m['dim'], m['vdim']
    for b in (1, 2):
      out[f'{p}norm{b}'] = norm(W)
      if case['family'] == 'hybrid':
        # (where tokens are chosen the embedding is to be seen behind the branches)
        out[f'{p}norm{b}b'] = norm(W) * (0.25 if case['kind'] == 'generate' else 1)
      else:
        out[f'{p}hc{b}.in'] = 1.0 / STREAMS + 0.1 * r.normal(STREAMS)
        out[f'{p}hc{b}.out'] = 1.0 + 0.1 * r.normal(STREAMS)
        out[f'{p}hc{b}.mix'] = (torch.eye(STREAMS, device=DEV) +
                                0.03 * r.normal(STREAMS, STREAMS))
    linear(q + 'o', W, H * Dv, small)
    if kind == 'attention':
      linear(q + 'q', H * D, W)
      linear(q + 'k', m['kv_heads'] * D, W)
      linear(q + 'v', m['kv_heads'] * Dv, W)
      out[q + 'q.norm'], out[q + 'k.norm'] = norm(D), norm(D)
      out[q + 'sink'] = r.normal(H)
    elif kind == 'latent_attention':
      linear(q + 'dq', m['q_rank'], W)
      out[q + 'dq.norm'] = norm(m['q_rank'])
      linear(q + 'uq', H * D, m['q_rank'])
      linear(q + 'uk', H * D, m['kv_rank'])
      linear(q + 'uv', H * Dv, m['kv_rank'])
      out[q + 'sink'] = r.normal(H)
      if m.get('kv_from') is None:
        linear(q + 'dkv', m['kv_rank'], W)
        out[q + 'dkv.norm'] = norm(m['kv_rank'])
    else:
      for name, n in (('q', H * D), ('k', H * D), ('v', H * Dv)):
        linear(q + name, n, W)
        if kind == 'channel_delta':
          out[f'{q}{name}.conv'] = 0.5 * r.normal(n, m['conv'])
      linear(q + 'a1', LOW, W)
      linear(q + 'a2', H * D, LOW)
      out[q + 'norm'] = norm(Dv)
      if kind == 'gla':
        linear(q + 'g', H * Dv, W)
        out[q + 'a2.b'] = 2.0 + 1.5 * r.normal(H * D)
      else:
        linear(q + 'b', H, W)
        linear(q + 'g1', LOW, W)
        linear(q + 'g2', H * Dv, LOW)
        out[q + 'A_log'] = 0.5 * r.normal(H)
        out[q + 'dt_bias'] = -3.0 + 1.5 * r.normal(H * D)
    if mlp['kind'] == 'dense':
      unit(p + 'mlp.', mlp['ff'])
    else:
      e = mlp['router']['experts']
      out[p + 'mlp.table'] = torch.rand(
          (VOCAB, e), generator=r.gen, device=DEV).argsort(1)[
              :, :mlp['router']['top']].to(torch.int32)
      for j in range(e):
        unit(f'{p}mlp.e{j}.', mlp['expert']['ff'])
      unit(p + 'mlp.shared.', mlp['shared']['ff'])
      linear(p + 'mlp.shared.sg', 1, W)
  return out


@functools.lru_cache(maxsize=1)  # a program loads its model once for all inputs
def _t5_model(size, dtype, decode):
  case = dict(size=size, dtype=dtype)
  params = _t5_params(case)
  cfg = network.t5_1_1_config(
      size, dtype='float32' if dtype == 'float32' else 'bfloat16',
      weight_dtype='int8' if dtype == 'int8' else None)
  module = network.Transformer(cfg)
  model = models.EncoderDecoderModel(
      module, decode_fn=(decoding.beam_search if decode == 'beam' else
                         decoding.temperature_sample))
  return model, params


@functools.lru_cache(maxsize=1)
def _lm_model(family, width, kind):
  case = dict(family=family, width=width, kind=kind)
  config = _lm_config(case)
  params = _lm_params(case, config)
  module = hybrid.HybridDecoder(hybrid.HybridConfig.from_dict(config, 'bfloat16'))
  module.decoder_weights(params)
  return models.DecoderOnlyModel(module), params


def _model_of(case):
  if 'size' in case:
    return _t5_model(case['size'], case.get('dtype', 'bfloat16'),
                     'beam' if case.get('beams') else 'sample')
  return _lm_model(case['family'], case['width'],
                   'generate' if case['kind'] == 'generate' else 'logits')


# ------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------


class Gumbel:
  """Sampling noise by step, from a seed."""

  def __init__(self, seed):
    self.seed = seed

  def noise(self, step, shape):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(self.seed * 4096 + int(step))
    u = torch.rand(shape, generator=gen, device=DEV)
    return -torch.log(-torch.log(u.clamp_min(1e-30)))


def _inputs(case, seed):
  """Host arrays, as a tokenizer or a request queue gives them."""
  rs = np.random.RandomState(seed % (1 << 31))
  text = lambda *s: rs.randint(2, VOCAB, size=s).astype(np.int32)
  kind = case['kind']
  if kind in ('predict', 'encode'):
    B, E = case['batch'], case['enc']
    tokens = text(B, E)
    lens = rs.randint(case['enc_min'], E + 1, size=B)
    tokens[np.arange(E)[None, :] >= lens[:, None]] = 0
    out = {'encoder_input_tokens': tokens}
    if kind == 'predict':
      # shifted right; the first target (a task's or language's tag) is given
      dec = np.zeros((B, case['length']), np.int32)
      dec[:, 1] = text(B)
      out['decoder_input_tokens'] = dec
    return out
  if kind == 'step':
    return {'ids': text(case['rows'])}
  B = case['batch']
  lens = rs.randint(case['shortest'], case['longest'] + 1, size=B)
  lens[rs.randint(B)] = case['longest']
  L = case['longest'] + case.get('new', 0)
  tokens = text(B, L) * (np.arange(L)[None, :] < lens[:, None])
  return {'tokens': tokens.astype(np.int32), 'lens': lens.astype(np.int32)}


def _fill_caches(case, config, leaves, seed):
  """What a cache holds in the middle of a sequence: keys and latents that have
  been normed, values, states of the size that the recurrences reach."""
  r = _Random(seed % (1 << 31) + 17, True)
  for run in sorted(leaves, key=lambda n: int(n.split('_')[1])):
    m = config['layers'][int(run.split('_')[1])]
    for name in sorted(leaves[run]):
      t = leaves[run][name]
      x = torch.randn(t.shape, generator=r.gen, device=DEV)
      if name == 'state':
        x *= 0.3 if m['type'] == 'channel_delta' else 2.0
      t.copy_(x)


def prepare(case, seed):
  model, params = _model_of(case)
  module, x = model.module, _inputs(case, seed)
  state = {'case': case, 'model': model, 'params': params, **x}
  if case['kind'] == 'predict':
    state['batch'] = {k: x[k] for k in ('encoder_input_tokens',
                                        'decoder_input_tokens')}
    state['noise'] = Gumbel(seed) if case['temperature'] else None
  elif case['kind'] == 'encode':
    state['encoder_input_tokens'] = torch.as_tensor(x['encoder_input_tokens'],
                                                    device=DEV)
  elif case['kind'] == 'prefill':
    B = case['batch']
    state['cache'] = module.init_cache(B, case['longest'] + 64)
    state['portions'] = [(r, 0, x['tokens'][r, :n]) for r, n in
                         enumerate(x['lens'])]
    state['want'] = [[n - 1] for n in x['lens']]
  elif case['kind'] == 'step':
    cache = module.init_cache(case['rows'], 4608, portion=64)
    _fill_caches(case, _lm_config(case), cache['decoder'], seed)
    cache['cache_index'].fill_(case['position'])
    state['cache'] = cache
    state['ids'] = torch.as_tensor(x['ids'], device=DEV)
  else:
    L = case['longest'] + case['new']
    state['batch'] = {
        'decoder_input_tokens': x['tokens'],
        'decoder_causal_attention': (np.arange(L)[None, :] <
                                     x['lens'][:, None]).astype(np.int32)}
  return state


def run(state):
  case, model, params = state['case'], state['model'], state['params']
  if case['kind'] == 'predict':
    options = {} if case['beams'] else {
        'temperature': case['temperature'], 'topk': case['topk'],
        'rescale_log_probs': False}
    tokens, aux = model.predict_batch_with_aux(
        params, state['batch'], rng=state['noise'], decoder_params=options,
        num_decodes=max(1, case['beams']), prompt_with_targets=True)
    return {'tokens': tokens, 'scores': aux['scores']}
  if case['kind'] == 'encode':
    return model.module.apply({'params': params}, state['encoder_input_tokens'],
                              enable_dropout=False, method=model.module.encode)
  if case['kind'] == 'prefill':
    logits = model.module.advance(params, state['cache'], state['portions'],
                                  state['want'])
    return {'logits': logits, 'cache': state['cache']['decoder']}
  if case['kind'] == 'step':
    logits = model.module.decode_step(params, state['cache'], state['ids'])
    return {'logits': logits, 'cache': state['cache']['decoder']}
  tokens, aux = model.predict_batch_with_aux(
      params, state['batch'],
      decoder_params={'temperature': 0.0, 'topk': 0, 'rescale_log_probs': False,
                      'max_decode_steps': case['new']})
  return {'tokens': tokens, 'scores': aux['scores']}


# ------------------------------------------------------------------------------
# Work
# ------------------------------------------------------------------------------


def _lm_weights(case):
  """(elements of the weights that every token passes, those of all experts,
  those of one)."""
  c, W = _lm_config(case), case['width']
  per_token = pool = one = 0
  for layer in c['layers']:
    m, mlp = layer['mixer'], layer['mlp']
    H, hd = m['heads'], m['heads'] * m['dim']
    per_token += hd * W
    if layer['type'] == 'attention':
      per_token += W * (hd + 2 * m['kv_heads'] * m['dim'])
    elif layer['type'] == 'latent_attention':
      per_token += m['q_rank'] * (W + hd) + 2 * RANK * hd
      per_token += 0 if m.get('kv_from') is not None else RANK * W
    else:
      low = 2 if layer['type'] == 'channel_delta' else 1
      per_token += W * (3 * hd + LOW * low) + low * LOW * hd
      per_token += W * (H if layer['type'] == 'channel_delta' else hd)
    if mlp['kind'] == 'dense':
      per_token += 3 * W * mlp['ff']
    else:
      per_token += 3 * W * mlp['shared']['ff']
      one += 3 * W * mlp['expert']['ff']
      pool += EXPERTS * 3 * W * mlp['expert']['ff']
  return per_token, pool, one


def _lm_work(case, lens, start, logits_rows):
  """One call over portions of these lengths that start at these positions."""
  per_token, pool, one = _lm_weights(case)
  c, W = _lm_config(case), case['width']
  M, S = sum(lens), len(lens)
  used = min(1.0, M * TOP / EXPERTS) if pool else 0.0
  flops = 2.0 * M * (per_token + TOP * one) + 2.0 * logits_rows * W * VOCAB
  bytes_ = 2.0 * (per_token + pool * used + W * VOCAB) + (
      4.0 * logits_rows * VOCAB + 2.0 * M * W)
  pairs = 0.0
  for n in lens:
    i = np.arange(start, start + n)
    pairs += float(np.minimum(i + 1, WINDOW).sum())
  kept = sum(min(start + n, WINDOW) - n for n in lens) if start else 0
  for layer in c['layers']:
    m = layer['mixer']
    hd = m['heads'] * m['dim']
    if layer['type'] == 'attention':
      flops += 4.0 * pairs * hd
      bytes_ += 4.0 * (kept + M) * m['kv_heads'] * m['dim']
    elif layer['type'] == 'latent_attention':
      flops += 4.0 * pairs * hd
      bytes_ += 2.0 * (kept + (M if m.get('kv_from') is None else 0)) * RANK
    else:
      flops += (7.0 if layer['type'] == 'channel_delta' else 5.0) * M * hd * HEAD
      bytes_ += (8.0 if start else 4.0) * S * hd * HEAD
  return bytes_, flops


def work(case):
  if 'size' in case:
    d, H, F, layers = T5[case['size']]
    hd = H * 64
    lens = (case['enc_min'] + case['enc']) / 2.0
    M = case['batch'] * lens
    s = 4 if case.get('dtype') == 'float32' else 2
    w = {'float32': 4, 'int8': 1}.get(case.get('dtype'), 2)
    per = 4 * d * hd + 3 * d * F  # weights of a layer's self-attention and MLP
    flops = layers * (2.0 * M * per + 4.0 * M * lens * hd)
    bytes_ = w * layers * per + 2.0 * s * M * d
    if case['kind'] == 'encode':
      return {'bytes': bytes_, 'flops': flops}
    R, L = case['batch'] * max(1, case['beams']), case['length']
    flops += layers * 4.0 * M * d * hd
    bytes_ += layers * 2.0 * w * d * hd
    # every step depends on the one before: it streams the decoder's weights, the
    # cross keys and values of every text and the self-attention cache
    step_w = layers * (per + 2 * d * hd) + d * VOCAB
    flops += L * (2.0 * R * step_w + layers * 4.0 * R * hd * (lens + L / 2.0))
    bytes_ += L * (w * step_w + layers * 2.0 * s * hd * (M + R * (L / 2.0 + 1)))
    return {'bytes': bytes_, 'flops': flops}
  if case['kind'] == 'step':
    bytes_, flops = _lm_work(case, [1] * case['rows'], case['position'],
                             case['rows'])
    return {'bytes': bytes_, 'flops': flops}
  mean = (case['longest'] + case['shortest']) // 2
  lens = [max(1, mean)] * case['batch']
  bytes_, flops = _lm_work(case, lens, 0,
                           case['batch'] if case['kind'] == 'prefill' else 0)
  if case['kind'] == 'generate':
    b, f = _lm_work(case, [1] * case['batch'], mean + case['new'] // 2,
                    case['batch'])
    bytes_, flops = bytes_ + case['new'] * b, flops + case['new'] * f
  return {'bytes': bytes_, 'flops': flops}


def tolerance(case):
  """About four times the distance from float64 that was measured over listed and
  drawn cases.  (Chosen tokens stand clear of the others, see _head.)"""
  kind, family = case['kind'], case.get('family')
  if kind == 'predict':
    if case['dtype'] == 'float32':  # 3e-7
      return {'rel': 2e-6, 'max': 1e-5, 'differ': 0.0}
    return {'rel': 0.025, 'max': 0.06, 'differ': 0.002}  # 0.006, 0.015
  if kind == 'generate':  # 0.0024, 0.0033
    return {'rel': 0.01, 'max': 0.015, 'differ': 0.002}
  if kind == 'encode':  # 0.013, 0.07
    return {'rel': 0.05, 'max': 0.25}
  if kind == 'step':  # 0.006, 0.04
    return {'rel': 0.025, 'max': 0.15}
  if family == 'latent':  # 0.0033, 0.06
    return {'rel': 0.013, 'max': 0.25}
  # 0.018; single entries of a state that a few tokens have written differ by more
  # than its root mean square
  return {'rel': 0.06}


# ------------------------------------------------------------------------------
# The same in float64
# ------------------------------------------------------------------------------


def _f64(t):
  return t.to(DEV).double()


def _rms(x):
  return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)


def _bucket(distance, bidirectional):
  """T5's buckets of key position - query position."""
  n, ret, buckets = -distance, 0, 32
  if bidirectional:
    buckets = 16
    ret = (n < 0).astype(np.int64) * buckets
    n = np.abs(n)
  else:
    n = np.maximum(n, 0)
  half = buckets // 2
  with np.errstate(divide='ignore'):
    far = half + (np.log(n.astype(np.float32) / half + np.finfo(np.float32).eps) /
                  np.log(128 / half) * (buckets - half)).astype(np.int32)
  return ret + np.where(n < half, n, np.minimum(far, buckets - 1))


class _T5Exact:

  def __init__(self, case):
    self.params = _model_of(case)[1]
    self.int8 = case.get('dtype') == 'int8'
    self.heads, self.layers = T5[case['size']][1], T5[case['size']][3]

  def kernel(self, p):
    w = p['kernel']
    if not self.int8:
      return _f64(w)
    scale = w.abs().amax(0).clamp_min(1e-30)
    scale = scale / torch.full_like(scale, 127.0)
    return _f64(torch.clamp(torch.round(w / scale), -127, 127)) * _f64(scale)

  def norm(self, x, p):
    return _rms(x) * _f64(p['scale'])

  def attend(self, p, xq, xkv, bias):
    B, Q, _ = xq.shape
    split = lambda t: t.view(B, -1, self.heads, 64).transpose(1, 2)
    q, k, v = (split(x @ self.kernel(p[n])) for x, n in (
        (xq, 'query'), (xkv, 'key'), (xkv, 'value')))
    out = torch.empty_like(q)
    step = max(1, (1 << 28) // max(1, self.heads * Q * k.shape[2]))
    for b in range(0, B, step):
      part = slice(b, b + step)
      s = q[part] @ k[part].transpose(2, 3)
      s = bias(s, part)
      out[part] = torch.softmax(s, -1) @ v[part]
    return out.transpose(1, 2).reshape(B, Q, -1) @ self.kernel(p['out'])

  def mlp(self, p, x):
    g = x @ self.kernel(p['wi_0'])
    g = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
    return (g * (x @ self.kernel(p['wi_1']))) @ self.kernel(p['wo'])

  def rel(self, p, Q, K, bidirectional):
    at = np.arange(K)[None, :] - np.arange(Q)[:, None]
    at = torch.as_tensor(_bucket(at, bidirectional), device=DEV)
    return _f64(p['relpos_bias']['rel_embedding'])[:, at]

  def encode(self, tokens):
    p = self.params['encoder']
    B, E = tokens.shape
    tokens = torch.nn.functional.pad(tokens, (0, -E % 4))  # (padded queries see it)
    rel = self.rel(p, tokens.shape[1], tokens.shape[1], True)
    valid = tokens > 0
    seen = valid[:, None, :, None] & valid[:, None, None, :]

    def bias(s, part):
      # a masked pair scores the same whatever its product: padding's own rows
      # weigh all positions alike
      return torch.where(seen[part], s + rel, torch.full_like(s, -1e10))

    x = _f64(self.params['token_embedder']['embedding'])[tokens]
    for i in range(self.layers):
      l = p[f'layers_{i}']
      h = self.norm(x, l['pre_attention_layer_norm'])
      x = x + self.attend(l['attention'], h, h, bias)
      x = x + self.mlp(l['mlp'], self.norm(x, l['pre_mlp_layer_norm']))
    return self.norm(x, p['encoder_norm'])[:, :E].contiguous()

  def logits(self, encoded, enc_tokens, ids):
    """Every position's logits of whole decoder sequences."""
    p = self.params['decoder']
    L = ids.shape[1]
    rel = self.rel(p, L, L, False)
    causal = torch.ones((L, L), dtype=torch.bool, device=DEV).tril()
    own = lambda s, part: torch.where(causal, s + rel, torch.full_like(s, -1e30))
    valid = (enc_tokens > 0)[:, None, None, :]
    cross = lambda s, part: torch.where(valid[part], s, torch.full_like(s, -1e30))
    x = _f64(self.params['token_embedder']['embedding'])[ids]
    for i in range(self.layers):
      l = p[f'layers_{i}']
      h = self.norm(x, l['pre_self_attention_layer_norm'])
      x = x + self.attend(l['self_attention'], h, h, own)
      h = self.norm(x, l['pre_cross_attention_layer_norm'])
      x = x + self.attend(l['encoder_decoder_attention'], h, encoded, cross)
      x = x + self.mlp(l['mlp'], self.norm(x, l['pre_mlp_layer_norm']))
    return self.norm(x, p['decoder_norm']) @ self.kernel(p['logits_dense'])


def _choose(case, logits, noise):
  """Tokens and their log-probabilities; noise: [rows, steps, VOCAB] or None."""
  logp = torch.log_softmax(logits, -1)
  if noise is not None:
    scaled = logits / case['temperature']
    least = torch.topk(scaled, case['topk'], -1).values[..., -1:]
    logits = torch.where(scaled >= least, scaled + noise,
                         torch.full_like(scaled, -1e30))
  tokens = logits.argmax(-1)
  return tokens, logp.gather(-1, tokens[..., None])[..., 0]


def _settle(tokens, found):
  """The next guess where `found` (what the model chooses after `tokens`) is not
  the guess itself: it holds up to a row's first difference, and on from there
  every token is followed by its successor."""
  after = torch.as_tensor(_successors(), device=DEV)
  n = tokens.shape[1]
  first = (tokens != found).int().argmax(1)
  out = torch.where(torch.arange(n, device=DEV)[None, :] <= first[:, None], found,
                    tokens)
  same = (tokens == found).all(1)
  for i in range(1, n):
    follow = (first < i) & ~same
    out[:, i] = torch.where(follow, after[out[:, i - 1]], out[:, i])
  return torch.where(same[:, None], tokens, out)


def _exact_predict(case, x, seed):
  e = _T5Exact(case)
  enc_tokens = torch.as_tensor(x['encoder_input_tokens'], device=DEV).long()
  dec = torch.as_tensor(x['decoder_input_tokens'], device=DEV).long()
  encoded = e.encode(enc_tokens)
  after = torch.as_tensor(_successors(), device=DEV)
  B, L = dec.shape
  ids = dec.clone()
  for i in range(2, L):
    ids[:, i] = after[ids[:, i - 1]]
  noise = None
  if case['temperature']:
    source = Gumbel(seed)
    noise = torch.stack([source.noise(i, (B, VOCAB)) for i in range(L)], 1)
  for _ in range(10):
    tokens, logp = _choose(case, e.logits(encoded, enc_tokens, ids), noise)
    tokens[:, 0] = dec[:, 1]
    if torch.equal(tokens[:, :-1], ids[:, 1:]):
      return {'tokens': tokens.int(), 'scores': logp[:, 1:].sum(1)}
    ids[:, 1:] = _settle(ids[:, 1:], tokens[:, :-1])
  return None


def _silu(x):
  return x * torch.sigmoid(x)


def _glu(h, w, p, limit, alpha, add):
  g = (h @ _f64(w[p + 'gate']).t()).clamp(max=limit)
  u = (h @ _f64(w[p + 'up']).t()).clamp(-limit, limit)
  return (g * torch.sigmoid(alpha * g) * (u + add)) @ _f64(w[p + 'down']).t()


class _LmExact:
  """tokens [B, T] (row b: lens[b] of them) at positions start ...; caches: what
  the model's cache tree holds before, by layer run, or None at the start."""

  def __init__(self, case):
    self.config = _lm_config(case)
    self.w = _model_of(case)[1]

  def __call__(self, tokens, lens, start=0, caches=None, rings=None):
    c, w = self.config, self.w
    W = c['width']
    self.B, self.T = tokens.shape
    self.lens, self.start = lens, start
    self.live = torch.arange(self.T, device=DEV)[None, :] < lens[:, None]
    self.caches, self.rings, self.left = caches, rings, {}
    x = _f64(w['embed'])[tokens]
    hyper = c['architecture'] == 'Nutizen'
    if hyper:
      x = x[None].repeat(c['streams'], 1, 1, 1)
    else:
      i = torch.arange((W + 1) // 2, device=DEV).double()
      pos = torch.arange(start, start + self.T, device=DEV).double()
      angle = pos[:, None] * torch.pow(torch.tensor(10000.0, device=DEV,
                                                    dtype=torch.float64),
                                       -2.0 * i / W)[None, :]
      wave = torch.zeros((self.T, W), dtype=torch.float64, device=DEV)
      wave[:, 0::2], wave[:, 1::2] = torch.sin(angle), torch.cos(angle)
      x = x + wave
    latents = {}
    for n, layer in enumerate(c['layers']):
      p = f'l{n}.'
      for b in (1, 2):
        norm = _f64(w[f'{p}norm{b}'])
        if hyper:
          h_in, h_mix, h_out = (_f64(w[f'{p}hc{b}.{k}']) for k in
                                ('in', 'mix', 'out'))
          h = _rms(torch.einsum('s,sbtw->btw', h_in, x)) * norm
        else:
          h = _rms(x) * norm
        y = (self.mix(n, layer, h, latents) if b == 1 else
             self.feed_forward(p + 'mlp.', layer['mlp'], h, tokens))
        if hyper:
          x = (torch.einsum('su,sbtw->ubtw', h_mix, x) +
               h_out[:, None, None, None] * y)
        else:
          x = x + _rms(y) * _f64(w[f'{p}norm{b}b'])
    return x.sum(0) if hyper else x

  def head(self, x):
    return (_rms(x) * _f64(self.w['final.norm'])) @ _f64(self.w['head']).t()

  def feed_forward(self, p, mlp, h, tokens):
    if mlp['kind'] == 'dense':
      if 'limit' in mlp:
        return _glu(h, self.w, p, mlp['limit'], 1.702, 1.0)
      return _glu(h, self.w, p, math.inf, 1.0, 0.0)
    out = torch.sigmoid(h @ _f64(self.w[p + 'shared.sg']).t()) * _glu(
        h, self.w, p + 'shared.', mlp['shared']['limit'], 1.702, 1.0)
    out, rows = out.view(-1, out.shape[-1]), h.reshape(-1, h.shape[-1])
    picks = self.w[p + 'table'].long()[tokens.reshape(-1)]
    for e in range(EXPERTS):
      at = (picks == e).any(1).nonzero()[:, 0]
      if len(at):
        out[at] += _glu(rows[at], self.w, f'{p}e{e}.', mlp['expert']['limit'],
                        1.702, 1.0) / TOP
    return out.view(h.shape)

  def mix(self, n, layer, h, latents):
    m, kind = layer['mixer'], layer['type']
    t = lambda name: _f64(self.w[f'l{n}.mix.{name}'])
    heads = lambda x, d: x.view(self.B, self.T, -1, d)
    D, Dv = m['dim'], m['vdim']
    if kind == 'attention':
      q = _rms(heads(h @ t('q').t(), D)) * t('q.norm')
      k = _rms(heads(h @ t('k').t(), D)) * t('k.norm')
      v = heads(h @ t('v').t(), Dv)
      k, v = (self.ring(n, name, x) for name, x in (('key_ring', k),
                                                    ('value_ring', v)))
      H = m['heads']
      slopes = 2.0 ** (-8.0 * (torch.arange(H, device=DEV).double() + 1) / H)
      o = self.attend(q, k, v, m['scale'], slopes, t('sink'))
    elif kind == 'latent_attention':
      q = heads((_rms(h @ t('dq').t()) * t('dq.norm')) @ t('uq').t(), D)
      if m.get('kv_from') is None:
        c = _rms(h @ t('dkv').t()) * t('dkv.norm')
        latents[n] = self.ring(n, 'latent_ring', c[:, :, None])[:, :, 0]
      c = latents[n if m.get('kv_from') is None else m['kv_from']]
      k, v = ((c @ t(name).t()).view(self.B, c.shape[1], -1, d)
              for name, d in (('uk', D), ('uv', Dv)))
      o = self.attend(q, k, v, m['scale'], None, t('sink'))
    else:
      o = self.recurrence(n, kind, m, h, t)
    return o.reshape(self.B, self.T, -1) @ t('o').t()

  def ring(self, n, name, x):
    """The entries that windows of the call can show, oldest first, and what the
    ring holds after it: x [B, T, G, d]."""
    if self.rings is None:
      return x
    ring = self.rings[f'run_{n}'][name]
    flat = ring.dim() == 3  # latents: one row per position
    old = _f64(ring)[:, None] if flat else _f64(ring)
    rows, T = old.shape[2], self.T
    back = min(self.start, WINDOW - 1)
    at = torch.arange(self.start - back, self.start, device=DEV) % rows
    prev = old[:, :, at].transpose(1, 2)
    for b in range(self.B):
      first = max(0, int(self.lens[b]) - rows)
      i = torch.arange(first, int(self.lens[b]), device=DEV)
      old[b][:, (self.start + i) % rows] = x[b, i].transpose(0, 1)
    self.left.setdefault(f'run_{n}', {})[name] = old[:, 0] if flat else old
    return torch.cat([prev, x], 1)

  def attend(self, q, k, v, scale, slopes, sink):
    """q [B, T, H, D] at the end of k, v [B, J, G, D]."""
    B, T, H, D = q.shape
    J, G = k.shape[1:3]
    rep = lambda x: x.repeat_interleave(H // G, 2).transpose(1, 2)
    q, k, v = q.transpose(1, 2), rep(k), rep(v)
    out = torch.empty((B, H, T, v.shape[3]), dtype=q.dtype, device=DEV)
    for i in range(0, T, 512):
      n = min(512, T - i)
      lo = max(0, J - T + i - WINDOW + 1)
      hi = J - T + i + n
      dist = (torch.arange(hi - n, hi, device=DEV)[:, None] -
              torch.arange(lo, hi, device=DEV)[None, :])
      s = q[:, :, i:i + n] @ k[:, :, lo:hi].transpose(2, 3) * scale
      if slopes is not None:
        s = s - slopes[:, None, None] * dist
      s = torch.where((dist >= 0) & (dist < WINDOW), s, torch.full_like(s, -1e30))
      s = torch.cat([s, sink[:, None, None].expand(B, H, n, 1)], 3)
      out[:, :, i:i + n] = torch.softmax(s, -1)[..., :-1] @ v[:, :, lo:hi]
    return out.transpose(1, 2)

  def recurrence(self, n, kind, m, h, t):
    B, T, H, D, Dv = self.B, self.T, m['heads'], m['dim'], m['vdim']
    heads = lambda x, d: x.view(B, T, H, d)
    delta = kind == 'channel_delta'
    raw = [h @ t(name).t() for name in ('q', 'k', 'v')]
    if delta:
      taps = m['conv']
      x = torch.cat(raw, 2)
      conv = torch.cat([t(name + '.conv') for name in ('q', 'k', 'v')])
      prev = torch.zeros((B, taps - 1, x.shape[2]), dtype=x.dtype, device=DEV)
      ring = None
      if self.caches is not None:
        ring = _f64(self.caches[f'run_{n}']['conv_ring'])
        at = torch.arange(self.start - taps + 1, self.start, device=DEV)
        prev = ring[:, at % taps] * (at >= 0)[None, :, None]
      whole = torch.cat([prev, x], 1)
      y = sum(whole[:, j:j + T] * conv[:, j] for j in range(taps))
      if self.rings is not None:
        if ring is None:
          ring = torch.zeros((B, taps, x.shape[2]), dtype=x.dtype, device=DEV)
        for b in range(B):
          ring[b, (self.start + int(self.lens[b]) - 1) % taps] = x[
              b, int(self.lens[b]) - 1]
        # (after a prompt the oldest of its rows is one that nothing reads)
        self.left.setdefault(f'run_{n}', {})['conv_ring'] = (
            ring if self.caches is not None else None)
      q, k, v = _silu(y).split([H * D, H * D, H * Dv], 2)
      unit = lambda x: x / torch.sqrt(x.square().sum(-1, keepdim=True) + 1e-6)
      q, k, v = unit(heads(q, D)) * D ** -0.5, unit(heads(k, D)), heads(v, Dv)
      beta = torch.sigmoid(h @ t('b').t())
      z = heads(h @ t('a1').t() @ t('a2').t() + t('dt_bias'), D)
      decay = torch.exp(-torch.exp(t('A_log'))[:, None] *
                        torch.nn.functional.softplus(z, threshold=60.0))
    else:
      q, k, v = heads(raw[0], D) * D ** -0.5, heads(raw[1], D), heads(raw[2], Dv)
      z = h @ t('a1').t() @ t('a2').t() + t('a2.b')
      decay = heads(torch.sigmoid(z).pow(1.0 / m['tau']), D)
    # what lies beyond a sequence's end leaves the state as it is
    live = self.live[:, :, None, None].double()
    decay, k = decay * live + (1 - live), k * live
    if self.caches is not None:
      S = _f64(self.caches[f'run_{n}']['state'])
    else:
      S = torch.zeros((B, H, D, Dv), dtype=h.dtype, device=DEV)
    o = torch.empty((B, T, H, Dv), dtype=h.dtype, device=DEV)
    for i in range(T):
      S = S * decay[:, i, :, :, None]
      u = v[:, i]
      if delta:
        u = beta[:, i, :, None] * (u - (k[:, i, :, None] @ S)[:, :, 0])
      S = S + k[:, i, :, :, None] * u[:, :, None, :]
      o[:, i] = (q[:, i, :, None] @ S)[:, :, 0]
    if self.rings is not None:
      self.left.setdefault(f'run_{n}', {})['state'] = S
    o = (_rms(o) * t('norm')).reshape(B, T, -1)
    if delta:
      return o * torch.sigmoid(h @ t('g1').t() @ t('g2').t())
    return o * _silu(h @ t('g').t())


def _exact_logits(case, x, seed):
  """Logits and cache after a prefill or a step."""
  e = _LmExact(case)
  state = prepare(case, seed)
  rings = state['cache']['decoder']  # (as they are before the call)
  if case['kind'] == 'step':
    tokens = torch.as_tensor(x['ids'], device=DEV).long()[:, None]
    lens = torch.ones(len(tokens), dtype=torch.long, device=DEV)
    hidden = e(tokens, lens, case['position'], rings, rings)
  else:
    tokens = torch.as_tensor(x['tokens'], device=DEV).long()
    lens = torch.as_tensor(x['lens'], device=DEV).long()
    hidden = e(tokens, lens, 0, None, rings)
  last = hidden[torch.arange(len(lens), device=DEV), lens - 1]
  return {'logits': e.head(last), 'cache': e.left}


def _exact_generate(case, x):
  e = _LmExact(case)
  after = torch.as_tensor(_successors(), device=DEV)
  lens = torch.as_tensor(x['lens'], device=DEV).long()
  # a row ends after the step at position lens + new - 1: new + 1 tokens
  ids = torch.nn.functional.pad(
      torch.as_tensor(x['tokens'], device=DEV).long(), (0, 1))
  B, L = ids.shape
  steps = case['new'] + 1
  at = lens[:, None] - 1 + torch.arange(steps, device=DEV)[None, :]
  tokens = torch.empty((B, steps), dtype=torch.long, device=DEV)
  tokens[:, 0] = after[ids.gather(1, at[:, :1])[:, 0]]
  for i in range(1, steps):
    tokens[:, i] = after[tokens[:, i - 1]]
  for _ in range(10):
    ids.scatter_(1, at + 1, tokens)
    hidden = e(ids, torch.full_like(lens, L))
    rows = hidden.gather(1, at[..., None].expand(-1, -1, hidden.shape[2]))
    found, logp = _choose(case, e.head(rows), None)
    if torch.equal(found, tokens):
      # column i is the token at position i + 1
      return {'tokens': ids[:, 1:].int(), 'scores': logp.sum(1)}
    tokens = _settle(tokens, found)
  return None


@torch.no_grad()
def exact(case, seed):
  x = _inputs(case, seed)
  if case['kind'] == 'predict':
    return _exact_predict(case, x, seed)
  if case['kind'] == 'encode':
    tokens = torch.as_tensor(x['encoder_input_tokens'], device=DEV).long()
    return _T5Exact(case).encode(tokens)
  if case['kind'] == 'generate':
    return _exact_generate(case, x)
  return _exact_logits(case, x, seed)
