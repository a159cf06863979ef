"""The fp16 logits' chain that reads and rounds halves inside its products (soft cap) against the oracle: caps that fp16 does not hold,
caps that saturate tanh or leave it linear, in both launch forms, on row lengths around the tile."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu
SIZES = [(1, 64), (63, 128), (65, 64), (200, 128), (321, 64), (520, 128)]
# A logit on a rounding boundary moves by one fp16 ulp, at most 2^-7 for logits below 16, and its probability by that share; outputs are
# means of values below 5 weighted by such probabilities, a few of which count: 5 * 2^-8, rounded up
O_BAR = 2e-2


@pytest.mark.parametrize("form", ["4", "8"])
@pytest.mark.parametrize("S,D", SIZES)
@pytest.mark.parametrize("cap", [33.3, 0.1, 1e4])
def test_soft_cap(monkeypatch, form, S, D, cap):
  q, k, v = oracle.prepare_inputs(2, S, 2, D, seed=S)
  q = q * 2
  monkeypatch.setenv("FT_ATTN_FORM", form)
  out = ops.gemma2(q.cuda(), k.cuda(), v.cuda(), softcap=cap)
  torch.cuda.synchronize()
  assert (out.float().cpu() - oracle.gemma2_forward(q, k, v, softcap=cap).float()).abs().max().item() <= O_BAR
