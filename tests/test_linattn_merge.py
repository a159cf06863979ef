"""The linear cores with the chunks folded in the output pass and with the separate launch, against the oracle: one chunk,
several, more than the eight that one round of folding takes (with few heads a chunk has four tiles of 128 tokens: nine
chunks from 4097 tokens on, seventeen from 8193 on), chunks of more than one tile, tokens one off a chunk, head_dim 32, every tensor type, q, k and
v as views."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fused", "launch"])
@pytest.mark.parametrize("B,S,H,D,dtype", [(1, 1, 1, 64, torch.float16), (2, 128, 2, 64, torch.bfloat16), (1, 129, 4, 32, torch.float16),
                                           (1, 1024, 2, 64, torch.float32), (1, 1025, 2, 64, torch.float16), (1, 4096, 1, 64, torch.float16),
                                           (1, 4097, 1, 64, torch.float16), (1, 5000, 2, 64, torch.float32), (2, 8193, 1, 64, torch.bfloat16), (1, 8200, 2, 32, torch.float16)])
def test_where_the_chunks_are_folded(gpu, monkeypatch, form, B, S, H, D, dtype):
  monkeypatch.setenv("FT_LINATTN_MERGE", form)
  q, k, v = oracle.prepare_inputs(B, S, H, D, seed=S, dtype=dtype)
  dev = [t.to(gpu) for t in (q, k, v)]
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  ref = oracle.ea_forward(q, k, v).float()
  assert (ops.ea(*dev).float().cpu() - ref).norm() <= tol * ref.norm()
  for normalize_q in (True, False):
    ref = oracle.sima_forward(q, k, v, normalize_q=normalize_q, out_dtype=torch.float32)
    out = ops.sima(*dev, normalize_q=normalize_q, out_dtype=torch.float32)
    assert (out.cpu() - ref).norm() <= tol * ref.norm()


@pytest.mark.parametrize("form", ["fused", "launch"])
@pytest.mark.parametrize("layout", ["packed", "bhsd", "longer"])
@pytest.mark.parametrize("B,S,H,dtype", [(2, 129, 2, torch.float16), (1, 4100, 2, torch.bfloat16), (2, 300, 4, torch.float32)])
def test_views(gpu, monkeypatch, form, layout, B, S, H, dtype):
  """q, k and v as parts of one projection's result, in [B, H, S, D] storage, as the head of longer sequences."""
  monkeypatch.setenv("FT_LINATTN_MERGE", form)
  q, k, v = oracle.prepare_inputs(B, S, H, 64, seed=S, dtype=dtype)
  if layout == "packed":
    dev = torch.cat([t.to(gpu) for t in (q, k, v)], 2).split(H, 2)
  elif layout == "bhsd":
    dev = [t.to(gpu).transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
  else:
    dev = [torch.cat([t.to(gpu), torch.full((B, 77, H, 64), 9.0, dtype=dtype, device=gpu)], 1)[:, :S] for t in (q, k, v)]
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  ref = oracle.ea_forward(q, k, v).float()
  assert (ops.ea(*dev).float().cpu() - ref).norm() <= tol * ref.norm()
  ref = oracle.sima_forward(q, k, v, out_dtype=torch.float32)
  assert (ops.sima(*dev, out_dtype=torch.float32).cpu() - ref).norm() <= tol * ref.norm()


@pytest.mark.parametrize("form", ["fused", "launch"])
@pytest.mark.parametrize("S,lost", [(40, [(0, 20)]), (700, [(0, 300), (512, 640)]), (4200, [(0, 1500), (2100, 2101), (4000, 4200)])])
@pytest.mark.parametrize("D,dtype,low", [(64, torch.float16, -torch.inf), (32, torch.float16, -60000.0), (64, torch.bfloat16, -torch.inf),
                                         (64, torch.float32, -torch.inf), (64, torch.float32, torch.finfo(torch.float32).min)])
def test_tokens_masked_in_k(gpu, monkeypatch, form, S, lost, D, dtype, low):
  """Padding masked with -inf or the type's lowest value in K (fp32 beyond fp16's range becomes -inf as it is loaded): whole strips,
  waves and chunks of it, in one channel only in the second head."""
  monkeypatch.setenv("FT_LINATTN_MERGE", form)
  q, k, v = oracle.prepare_inputs(1, S, 2, D, seed=S, dtype=dtype)
  for a, b in lost:
    k[:, a:b, 0], k[:, a:b, 1, 3] = low, low
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  ref = oracle.ea_forward(q, k, v).float()
  out = ops.ea(q.to(gpu), k.to(gpu), v.to(gpu)).float().cpu()
  assert ref.isfinite().all() and (out - ref).norm() <= tol * ref.norm()
