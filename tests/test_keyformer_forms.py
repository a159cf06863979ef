"""KeyFormer's launch forms (128-row, 256-row and two-team workgroups of the attention pass, one and two teams of the column
pass) on noise rows of every alignment, against the oracle: row lengths around the tile, odd strides, noise from a seed."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu
FORMS = [("4", "2"), ("8", "2"), ("t", "1t")]


def _score_bar(S, dtype):
  # a logit on a rounding boundary moves one probability by up to an ulp (fp16 2^-10, bf16 2^-7 relative, times |logit|),
  # which a key seen by n rows shows as 1/n of it
  n = torch.arange(S, 0, -1, dtype=torch.float32)
  return (1e-3 + 4e-3 / n) if dtype == torch.float16 else (8e-3 + 3.2e-2 / n)


def _check(out, score, ref_out, ref_score, dtype):
  assert (out.float().cpu() - ref_out.float()).abs().max().item() <= 2e-2
  rel = ((score.cpu() - ref_score).abs() / ref_score).amax(dim=(0, 1))
  assert (rel <= _score_bar(rel.numel(), dtype)).all(), rel.max().item()


@pytest.mark.parametrize("form,keys", FORMS)
@pytest.mark.parametrize("S,D,pad,dtype", [
    (1, 64, 0, torch.float16), (3, 128, 0, torch.float16), (64, 64, 0, torch.float16), (65, 128, 0, torch.float16),
    (130, 128, 0, torch.bfloat16), (190, 64, 1, torch.float16), (192, 128, 4, torch.float16), (257, 128, 0, torch.float16),
    (323, 64, 2, torch.bfloat16), (450, 128, 3, torch.float16)])
def test_noise_tensor(monkeypatch, form, keys, S, D, pad, dtype):
  q, k, v = oracle.prepare_inputs(2, S, 3, D, seed=S, dtype=dtype)
  er = oracle.prepare_exp_rand(2, 3, S, S + pad, seed=S)[..., :S]
  monkeypatch.setenv("FT_ATTN_FORM", form)
  monkeypatch.setenv("FT_COLSTATS_KEYS", keys)
  dev_er = torch.empty(2, 3, S, S + pad, device="cuda").fill_(float("nan"))[..., :S]
  dev_er.copy_(er)
  out, score = ops.keyformer(q.cuda(), k.cuda(), v.cuda(), dev_er, tau=1.5)
  torch.cuda.synchronize()
  _check(out, score, *oracle.keyformer_forward(q, k, v, er.contiguous(), tau=1.5), dtype)


@pytest.mark.parametrize("tau", [1.0, 0.6, 0.2])  # the packed forms, and the generic one below a quarter
@pytest.mark.parametrize("S,D,dtype", [(65, 128, torch.float16), (200, 64, torch.float16), (321, 128, torch.float16), (256, 64, torch.bfloat16)])
def test_seeded_noise_two_teams(monkeypatch, tau, S, D, dtype):
  q, k, v = (x.cuda() for x in oracle.prepare_inputs(2, S, 3, D, seed=S, dtype=dtype))
  got = {}
  for form in ("4", "t"):
    monkeypatch.setenv("FT_ATTN_FORM", form)
    got[form] = ops.keyformer(q, k, v, None, tau=tau, seed=11)
  torch.cuda.synchronize()
  # results below 4 and one ulp apart: 2^-9 in fp16, 2^-6 in bf16
  assert (got["t"][0].float() - got["4"][0].float()).abs().max().item() <= (2**-9 if dtype == torch.float16 else 2**-6)
  # fp32 sums of up to S terms in another order, and through the exponential of the normaliser: S 2^-24 / tau
  torch.testing.assert_close(got["t"][1], got["4"][1], rtol=max(2e-5, 4 * S * 2**-24 / tau), atol=0)


@pytest.mark.parametrize("form", ["4", "8", "t"])
def test_noise_rows_far_apart(monkeypatch, form):
  """Rows of the noise tensor 128 MiB apart: beyond what a 32-bit offset from a wave's first row reaches."""
  S, D = 67, 64
  q, k, v = oracle.prepare_inputs(1, S, 1, D, seed=5)
  er = oracle.prepare_exp_rand(1, 1, S, S, seed=5)
  far = torch.empty(0, device="cuda").set_(torch.empty((S - 1) * 2**25 + S, device="cuda").untyped_storage(), 0, (1, 1, S, S), (0, 0, 2**25, 1))
  far.copy_(er)
  monkeypatch.setenv("FT_ATTN_FORM", form)
  out, score = ops.keyformer(q.cuda(), k.cuda(), v.cuda(), far, tau=1.5)
  torch.cuda.synchronize()
  _check(out, score, *oracle.keyformer_forward(q, k, v, er, tau=1.5), torch.float16)
