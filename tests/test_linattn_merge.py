"""The linear cores with the chunks folded in the output pass and with the separate launch, against the oracle: one chunk,
several, chunks of more than one tile, tokens one off a chunk, head_dim 32, every tensor type."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fused", "launch"])
@pytest.mark.parametrize("B,S,H,D,dtype", [(1, 1, 1, 64, torch.float16), (2, 128, 2, 64, torch.bfloat16), (1, 129, 4, 32, torch.float16),
                                           (1, 1024, 2, 64, torch.float32), (1, 1025, 2, 64, torch.float16), (1, 4096, 1, 64, torch.float16)])
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
