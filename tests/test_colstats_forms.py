"""The column pass with 64 and with 128 keys per workgroup and with 64 keys and two teams of waves: the forms
agree up to the order of fp32 sums; all are checked against the oracle."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,Skv,D,dtype,causal", [
    (1, 1, 128, torch.float16, True), (63, 63, 64, torch.float16, True), (65, 65, 128, torch.float16, False), (40, 129, 128, torch.bfloat16, True),
    (321, 321, 128, torch.float16, True), (513, 700, 128, torch.float16, True), (128, 128, 128, torch.bfloat16, False),
    (200, 450, 64, torch.bfloat16, False), (700, 700, 64, torch.float16, True)])
def test_forms(gpu, monkeypatch, Sq, Skv, D, dtype, causal):
  q, k, v = oracle.prepare_inputs(1, Sq, 2, D, seed=Sq, dtype=dtype, kv_len=Skv)
  dev = [t.to(gpu) for t in (q, k, v)]
  res = {}
  monkeypatch.setenv("FT_ATTN_FORM", "4")  # the column pass whatever the number of rows
  for form in ("1", "2", "1t"):
    monkeypatch.setenv("FT_COLSTATS_KEYS", form)
    res[form] = [*ops.roco(*dev, causal=causal), ops.h2o(*dev, causal=causal)[1], *ops.corm(*dev, causal=causal, return_margin=True)[1:],
                 *(ops.keyformer(*dev, None, tau=t, seed=3, causal=causal)[1] for t in (1.0, 1.5, 0.2))]
  for other in (res["2"], res["1t"]):
    for a, b in zip(res["1"], other):
      assert torch.allclose(a.float(), b.float(), rtol=1e-5, atol=1e-6)
  if causal:
    _, r1, r2 = oracle.roco_forward(q, k, v)
    tol = 1e-2 if dtype is torch.bfloat16 else 1e-3
    for r in res.values():
      assert (r[1].cpu() - r1).norm() <= tol * r1.norm() and (r[2].cpu() - r2).norm() <= 2 * tol * r2.norm()
