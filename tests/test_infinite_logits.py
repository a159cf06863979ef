"""Keys whose product with a query leaves the range of the tensor type: their logits are -inf and their probability 0
(the reference's rounded QK^T), wherever they fall in a row's key tiles: its first ones, a whole share or the first tile of
one, a share of a single key.  A row all of whose visible keys are such has no softmax: the reference's result is NaN there."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


def _inputs(Sq, Skv, H, D, dtype, lost):
  """N(0, 1) but for four channels, whose product is far below the lowest finite value for the keys in `lost`, 0 for others."""
  q, k, v = oracle.prepare_inputs(1, Sq, H, D, seed=Sq + Skv, dtype=dtype, kv_len=Skv)
  big = 2e19 if dtype is torch.bfloat16 else 200.0  # 4 * 2e19**2 = 1.6e39 > 3.4e38, 4 * 200**2 = 160 000 > 65 504
  q[..., :4], k[..., :4] = big, 0
  for a, b in lost:
    k[:, a:b, :, :4] = -big
  return q, k, v


def _close(got, ref, tol, what):
  """NaN exactly where the reference has it, and of the rest the norm of the difference."""
  got, ref = got.float().cpu(), ref.float()
  assert torch.equal(got.isnan(), ref.isnan()), f"{what}: {got.isnan().sum()} NaN, reference {ref.isnan().sum()}"
  got, ref = got.nan_to_num(0.0), ref.nan_to_num(0.0)
  assert (got - ref).norm() <= tol * ref.norm(), what


# key ranges that are lost; with a causal mask the rows that see nothing else are NaN
@pytest.mark.parametrize("form", ["", "s1", "s3", "t", "4", "8"])
@pytest.mark.parametrize("Sq,Skv,lost", [
    (1, 65, [(64, 65)]),                              # the last share is one lost key
    (1, 449, [(0, 64)]),                              # the row's first tile
    (8, 700, [(0, 5), (64, 128), (192, 400)]),        # whole shares, and a tile that is also a share's first
    (33, 640, [(192, 256)]),                          # the first tile of the second share of three tiles
    (65, 65, [(64, 65)]),                             # the second team's only key
    (300, 300, [(64, 193)]), (300, 300, [(0, 40)]),   # rows with nothing left: NaN
    (130, 1090, [(0, 70), (500, 600), (1088, 1090)])])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.float16), (64, torch.bfloat16), (128, torch.bfloat16)])
def test_keys_below_the_range(gpu, monkeypatch, form, Sq, Skv, lost, D, dtype):
  monkeypatch.setenv("FT_ATTN_FORM", form)
  q, k, v = _inputs(Sq, Skv, 2, D, dtype, lost)
  dev = [t.to(gpu) for t in (q, k, v)]
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  ref_o, ref_s, ref_sq = oracle.roco_forward(q, k, v)
  out, s, sq = ops.roco(*dev)
  _close(out, ref_o, tol, "out")
  seen = ~ref_s.isnan()  # a row of NaN makes every sum over it NaN in the reference; keys it does not see may keep theirs here
  _close(s.cpu().where(seen, torch.nan), ref_s, tol, "sums")
  _close(sq.cpu().where(seen, torch.nan), ref_sq, 2 * tol, "squares")
  _close(ops.attn(*dev), ref_o, tol, "attn")


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.float16), (64, torch.bfloat16)])
@pytest.mark.parametrize("tau", [1.0, 1.5, 0.2])
def test_keys_below_the_range_under_noise(gpu, D, dtype, tau):
  """The perturbed softmax's own maximum, and the plain one's that the packed forms share."""
  q, k, v = _inputs(40, 200, 2, D, dtype, [(0, 70), (130, 131)])
  dev = [t.to(gpu) for t in (q, k, v)]
  tol = 1e-2 if dtype is torch.bfloat16 else 4e-3
  for seed, er in ((5, oracle.seeded_exp_rand(5, 1, 2, 40, 200)), (None, oracle.prepare_exp_rand(1, 2, 40, 200, seed=1))):
    ref_o, ref_s = oracle.keyformer_forward(q, k, v, er, tau)
    out, s = ops.keyformer(*dev, er.to(gpu) if seed is None else None, tau=tau, seed=seed or 0)
    _close(out, ref_o, tol, "out")
    _close(s, ref_s, tol, "score")


@pytest.mark.parametrize("form", ["", "s1", "s2", "t", "4"])
@pytest.mark.parametrize("Sq,Skv,D,dtype", [(1, 200, 128, torch.float16), (6, 333, 64, torch.float16), (40, 260, 128, torch.float16), (3, 300, 64, torch.bfloat16)])
def test_keys_below_the_range_under_groups(gpu, monkeypatch, form, Sq, Skv, D, dtype):
  """Two batches, four query heads on each of two k/v heads; the two k/v heads lose different keys."""
  monkeypatch.setenv("FT_ATTN_FORM", form)
  B, H, Hkv = 2, 8, 2
  q, k, v = oracle.prepare_inputs(B, Sq, H, D, seed=Skv, dtype=dtype, kv_len=Skv)
  k, v = k[:, :, :Hkv].contiguous(), v[:, :, :Hkv].contiguous()
  big = 2e19 if dtype is torch.bfloat16 else 200.0
  q[..., :4], k[..., :4] = big, 0
  k[:, :65, 0, :4], k[:, 128:192, 1, :4], k[1, Skv - 1, 1, :4] = -big, -big, -big
  kr, vr = (t.repeat_interleave(H // Hkv, 2) for t in (k, v))
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  ref_o, ref_s = oracle.h2o_forward(q, kr, vr)
  out, score = ops.h2o(*(t.to(gpu) for t in (q, k, v)))
  _close(out, ref_o, tol, "out")
  _close(score, ref_s.view(B, Hkv, H // Hkv, Skv).mean(2), tol, "sums")
