"""The column pass with 64 and with 128 keys per workgroup: a key is summed over the same rows in the same order; one
form is checked against the oracle."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,Skv,D,dtype,causal", [
    (1, 1, 128, torch.float16, True), (63, 63, 64, torch.float16, True), (65, 65, 128, torch.float16, False), (40, 129, 128, torch.bfloat16, True),
    (321, 321, 128, torch.float16, True), (200, 450, 64, torch.bfloat16, False), (700, 700, 64, torch.float16, True)])
def test_both_forms(gpu, monkeypatch, Sq, Skv, D, dtype, causal):
  q, k, v = oracle.prepare_inputs(1, Sq, 2, D, seed=Sq, dtype=dtype, kv_len=Skv)
  dev = [t.to(gpu) for t in (q, k, v)]
  res = {}
  monkeypatch.setenv("FT_ATTN_FORM", "4")  # the column pass whatever the number of rows
  for keys in ("1", "2"):
    monkeypatch.setenv("FT_COLSTATS_KEYS", keys)
    res[keys] = [*ops.roco(*dev, causal=causal), ops.h2o(*dev, causal=causal)[1], *ops.corm(*dev, causal=causal, return_margin=True)[1:],
                 *(ops.keyformer(*dev, None, tau=t, seed=3, causal=causal)[1] for t in (1.0, 1.5, 0.2))]
  for a, b in zip(*res.values()):
    assert torch.allclose(a.float(), b.float(), rtol=1e-5, atol=1e-6)
  if causal:
    _, r1, r2 = oracle.roco_forward(q, k, v)
    tol = 1e-2 if dtype is torch.bfloat16 else 1e-3
    assert (res["1"][1].cpu() - r1).norm() <= tol * r1.norm() and (res["1"][2].cpu() - r2).norm() <= 2 * tol * r2.norm()
