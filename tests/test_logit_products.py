"""The fp16 logits' chains that read and round halves inside their products (soft cap, KeyFormer with noise from a tensor) against
the oracle: caps that fp16 does not hold, caps that saturate tanh or leave it linear, temperatures on both sides of 1, in every
launch form, on row lengths around the tile."""
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


@pytest.mark.parametrize("form", ["4", "8", "t"])
@pytest.mark.parametrize("S,D", SIZES)
@pytest.mark.parametrize("tau", [0.5, 4.0])
def test_keyformer_tensor(monkeypatch, form, S, D, tau):
  q, k, v = oracle.prepare_inputs(2, S, 2, D, seed=S)
  er = oracle.prepare_exp_rand(2, 2, S, S, seed=S)
  monkeypatch.setenv("FT_ATTN_FORM", form)
  out, score = ops.keyformer(q.cuda(), k.cuda(), v.cuda(), er.cuda(), tau=tau)
  torch.cuda.synchronize()
  ref_out, ref_score = oracle.keyformer_forward(q, k, v, er, tau=tau)
  assert (out.float().cpu() - ref_out.float()).abs().max().item() <= O_BAR
  # one ulp of a logit below 4 (2^-9) moves a probability by that share over tau, and a key seen by n rows by 1 / n of it
  n = torch.arange(S, 0, -1, dtype=torch.float32)
  rel = ((score.cpu() - ref_score).abs() / ref_score).amax(dim=(0, 1))
  assert (rel <= (1e-3 + 4e-3 / n) / min(tau, 1.0)).all(), rel.max().item()
