"""The C-ABI library loads and exports every entry point include/*.h
declare (no compute calls: this runs without a GPU)."""

import ctypes
import os
import re

import pytest

from t5x_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_names():
  inc = os.path.join(ROOT, 'include')
  text = ''.join(open(os.path.join(inc, f)).read()
                 for f in sorted(os.listdir(inc)) if f.endswith('.h'))
  text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
  return sorted(set(re.findall(r'\b(t5d_[a-z0-9_]+)\s*\(', text)))


def test_header_declares_entry_points():
  names = declared_names()
  assert 't5d_gemm' in names and 't5d_self_attention_step' in names
  assert len(names) >= 18


def test_library_exports_every_declared_symbol():
  if not os.path.exists(_lib.LIB_PATH):
    pytest.fail(f'{_lib.LIB_PATH} not built: run __graft_entry__.build()')
  lib = ctypes.CDLL(_lib.LIB_PATH)
  missing = [n for n in declared_names() if not hasattr(lib, n)]
  assert not missing, missing


def test_binding_covers_every_declared_symbol():
  assert set(declared_names()) == set(_lib.exported_names())


def test_binding_names_each_symbol_once():
  text = open(os.path.join(ROOT, 't5x_amd', '_lib.py')).read()
  names = re.findall(r"^    '(t5d_[a-z0-9_]+)': \(", text, flags=re.M)
  assert set(names) == set(_lib._SIGNATURES) and len(names) == len(set(names))


def test_measurement_aids_stay_out_of_the_boundary():
  """The work-skipping switch bench.py uses lives in its own header and entry
  point; the boundary's structs and declarations carry none."""
  boundary = open(os.path.join(ROOT, 'include', 't5d.h')).read()
  assert 'leave_out' not in boundary and 'LEAVE_OUT' not in boundary
  aids = open(os.path.join(ROOT, 'include', 't5d_measure.h')).read()
  assert 't5d_measure_leave_out' in aids
  if not os.path.exists(_lib.LIB_PATH):
    pytest.fail(f'{_lib.LIB_PATH} not built: run __graft_entry__.build()')
  assert hasattr(ctypes.CDLL(_lib.LIB_PATH), 't5d_measure_leave_out')
  assert _lib.measure_leave_out(0) == 0
  # no product module calls it
  pkg = os.path.join(ROOT, 't5x_amd')
  users = [f for f in os.listdir(pkg) if f.endswith('.py') and
           'measure_leave_out(' in open(os.path.join(pkg, f)).read()]
  assert sorted(users) == ['_lib.py', 'network.py']  # iteration_graph only


def test_static_entry_point_calls_no_allocator():
  """Source check: neither the entry point nor its address look-up names an
  allocating or freeing HIP call."""
  src = open(os.path.join(ROOT, 't5x_amd', 'csrc', 'select.hip')).read()
  start = src.index('static int static_topk_scratch(')
  entry = src.index('extern "C" int t5d_beam_topk_static(')
  end = src.index('\n}\n', entry)
  body = src[start:end]
  assert 'hipGetSymbolAddress' in body
  assert not re.search(r'hipMalloc|hipFree|hipMallocAsync|hipHostMalloc|'
                       r'hipExtMalloc|hipMemPool', body)


def test_version_and_error_string_without_gpu():
  lib = _lib.load()
  assert lib.t5d_version() == 1
  # shape validation happens on the host before any launch
  assert lib.t5d_packed_weight_bytes(_lib.BF16, 768, 2304) == 768 * 2304 * 2
  assert lib.t5d_packed_weight_bytes(_lib.I8, 768, 2304) == 768 * 2304
  assert lib.t5d_packed_weight_bytes(_lib.BF16, 40, 32) == -1
  rc = lib.t5d_rmsnorm(None, 7, None, None, None, 1, 1, 1e-6)
  assert rc == -1
  assert b'dtype' in lib.t5d_last_error()


def test_encoder_attention_beyond_a_launch_grid_without_gpu():
  """More tiles than one dimension of a grid holds are named, not left to the launch
  (the buffers are not looked at before)."""
  from t5x_amd import _lib
  lib = _lib.load()
  p, H = 4096, 300
  rc = lib.t5d_encoder_attention_variant(None, p, p, p, p, p, None, p, 65535, H, 100,
                                         128, H * 64, H * 64, 0)
  assert rc == -3  # T5D_ELIMIT
  assert b'launch grid' in lib.t5d_last_error()


@pytest.mark.parametrize('B,E', [(1, 2049), (1 << 19, 1), (1 << 20, 1023), (525000, 2046)])
def test_encoder_rows_beyond_their_numbers_without_gpu(B, E):
  """What t5d_encoder_rows names as too much, the encoder does not ask of it (it computes
  every position then)."""
  from t5x_amd import ops
  assert _lib.load().t5d_encoder_rows(None, 16, B, E, *[16] * 7) == -3  # T5D_ELIMIT
  assert not ops.EncoderRows.covers(B, E)
  for there in ((1, 2048), ((1 << 19) - 1, 2044), (32, 512)):
    assert ops.EncoderRows.covers(*there) == (there[0] * there[1] < 1 << 30)


@pytest.mark.parametrize('M,ld,N,one', [
    # widths that fill the kernel's variants, whatever the columns
    (4, 512, 131072, 1), (4, 1024, 131072, 1), (4, 1536, 131072, 1), (4, 2048, 131072, 1),
    (1, 64, 131072, 1), (2, 128, 50304, 1), (2, 64, 131072, 0),
    # few weights per workgroup
    (3, 64, 4096, 1), (3, 64, 32128, 0), (4, 256, 32128, 1), (4, 256, 50304, 0),
    (4, 384, 24576, 1), (4, 384, 32128, 0), (2, 384, 131072, 1),
    # the variant of 2048 inputs at a little over 1024
    (4, 1088, 16384, 1), (3, 1152, 32128, 0), (4, 1408, 24576, 0), (2, 1088, 32128, 1),
    (2, 1088, 50304, 0), (2, 1280, 131072, 1), (1, 1088, 50304, 1), (1, 1088, 131072, 0)])
def test_where_the_row_kernel_and_the_layer_behind_it_go_in_one_launch(M, ld, N, one):
  """t5d_stream_dense_pays: not where the two launches were measured to be faster."""
  from t5x_amd import _lib
  assert _lib.load().t5d_stream_dense_pays(M, ld, N) == one


# (float32 rows may lie anywhere, with any number of columns)
_BOTH = [dict(low_n=528), dict(off_z=320), dict(off_z=-16), dict(off_low_gate=320),
         dict(off_low_gate=-16), dict(off_low=1736), dict(off_low=-8), dict(low_k=0),
         dict(ld_low=304)]
_BF16 = [dict(low=8), dict(low_w=8), dict(low_n=558, ld_low=560)]


@pytest.mark.parametrize('dtype,wrong', [(_lib.F32, w) for w in _BOTH] +
                         [(_lib.BF16, w) for w in _BOTH + _BF16])
@pytest.mark.parametrize('rows', [1, 40])
def test_low_rank_columns_that_are_not_there_without_gpu(rows, dtype, wrong):
  """t5d_recurrence_run with low_w refuses sizes beyond its columns and what t5d_dense
  refuses, whichever of them would form the columns."""
  r = _lib.Recurrence()
  r.dtype, r.H, r.G, r.D, r.Dv = dtype, 4, 4, 64, 64
  r.delta = r.decay = r.unit = r.gate = 1
  for name in ('proj', 'low', 'decay_bias', 'A_log', 'norm', 'state', 'out', 'workspace',
               'low_w'):
    setattr(r, name, 4096)
  r.ld_proj, r.ld_out, r.workspace_bytes = 1664, 256, 1 << 40
  r.off_q, r.off_k, r.off_v, r.off_beta, r.off_gate = 0, 256, 512, 768, 1024
  r.off_low, r.low_k, r.low_n, r.ld_low = 1536, 128, 560, 560
  r.off_z, r.off_low_gate = 16, 288
  for name, value in wrong.items():
    setattr(r, name, value)
  b = _lib.Ragged()
  b.M = b.max_len = rows
  b.S = 1
  for name in ('tokens', 'tok_pos', 'tok_seq', 'seq_off', 'seq_start', 'seq_slot'):
    setattr(b, name, 4096)
  lib = _lib.load()
  assert lib.t5d_recurrence_run(None, ctypes.byref(r), ctypes.byref(b), 0) == -1
  assert b'low-rank' in lib.t5d_last_error() or b't5d_dense' in lib.t5d_last_error()


@pytest.mark.parametrize('M,ld,N,one', [
    # columns that fit 256 workgroups, and not
    (16, 512, 32768, 1), (16, 512, 32784, 0), (128, 768, 4096, 1), (128, 768, 4112, 0),
    # beyond 768 inputs more than one column tile per CU, and of four tiles more than 192
    # workgroups
    (16, 1024, 4096, 0), (16, 1024, 4112, 1), (33, 1024, 5632, 1), (64, 1024, 5632, 1),
    (33, 896, 8192, 0), (64, 896, 8192, 1), (96, 1024, 4096, 0), (112, 1024, 3328, 1),
    (112, 1024, 4096, 1),
    # few inputs, three and four tiles
    (33, 64, 8192, 0), (33, 192, 8192, 1), (80, 128, 4608, 0), (80, 128, 3072, 1)])
def test_where_the_row_kernel_and_a_layer_of_more_rows_go_in_one_launch(M, ld, N, one):
  """t5d_stream_rows_dense_pays: not where the two launches were measured to be faster."""
  assert _lib.load().t5d_stream_rows_dense_pays(M, ld, N) == one


@pytest.mark.parametrize('name', ['proj', 'cq', 'q', 'uq', 'ql', 'ol', 'latent_ring'])
@pytest.mark.parametrize('rows', [1, 200])
def test_latent_operands_off_16_bytes_without_gpu(rows, name):
  """t5d_latent_attention_run refuses them before it launches anything, whether the queries'
  layer goes alone or with the latents' norms."""
  a = _lib.LatentAttention()
  a.dtype, a.H, a.D, a.Dv, a.rank, a.q_rank = _lib.BF16, 4, 64, 64, 128, 256
  a.ring, a.ld_proj, a.off_q, a.off_kv, a.ld_out = 256, 512, 0, 256, 256
  for p in ('proj', 'q_norm', 'kv_norm', 'uq', 'absorb', 'expand', 'latent_ring', 'cq', 'q',
            'ql', 'ol', 'out'):
    setattr(a, p, 4096 + 8 * (p == name))
  b = _lib.Ragged()
  b.M = b.max_len = rows
  b.S = 1
  for p in ('tokens', 'tok_pos', 'tok_seq', 'seq_off', 'seq_start', 'seq_slot'):
    setattr(b, p, 4096)
  lib = _lib.load()
  assert lib.t5d_latent_attention_run(None, ctypes.byref(a), ctypes.byref(b), 0) == -1
  assert b'operand alignment' in lib.t5d_last_error()


def test_many_row_tile_choice_without_gpu():
  """t5d_gemm_rows_tile: which workgroup tile the many-row dense kernel runs a
  shape on (1: 128 columns, 2: 256, 3: 192, each of 128 rows, or 1 of 64), by what
  rounds of workgroups on 256 CUs cost.  The T5.1.1-base encoder over 32 x 512
  positions:"""
  lib = _lib.load()
  pick = lambda M, K, N, w=_lib.BF16: lib.t5d_gemm_rows_tile(w, M, K, N)
  assert pick(16384, 768, 768) == 3     # 512 tiles of 192 columns, two per CU
  assert pick(16384, 2048, 768) == 3
  assert pick(16384, 768, 4096) == 2    # 4 full rounds of 512 tiles of 256 columns
  assert pick(16384, 768, 1536) == 3    # 2 full rounds of 512 tiles of 192
  assert pick(16384, 4096, 4096) == 2
  assert pick(300, 96, 80) == 1         # one small workgroup
  # not chosen: int8 weights have 128 columns, K < 64 the staging-register kernel
  assert pick(16384, 768, 768, _lib.I8) == 1
  assert pick(16384, 32, 768) == 1


def test_product_path_has_no_cpu_fallback():
  import torch
  if torch.cuda.is_available():
    pytest.skip('GPU present')
  from t5x_amd import decoding
  with pytest.raises(RuntimeError, match='no CPU fallback'):
    decoding.beam_search([[0, 0]], {}, lambda s: None, 1)


def test_product_does_not_import_oracle():
  pkg = os.path.join(ROOT, 't5x_amd')
  for dirpath, _, files in os.walk(pkg):
    for f in files:
      if f.endswith('.py'):
        src = open(os.path.join(dirpath, f)).read()
        assert not re.search(r'^\s*(from|import)\s+oracle\b', src, re.M), f
