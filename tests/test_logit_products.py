"""The fp16 logits' chains whose products read halves by themselves (soft cap, KeyFormer with noise from a tensor) against the oracle:
caps that fp16 does not hold, caps that saturate tanh or leave it linear, temperatures on both sides of 1, on row lengths around the
tile and over longer keys of fewer heads, in each launch form of the attention pass; and the places where they round."""
import math

import numpy as np
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu
SIZES = [(1, 64), (63, 128), (65, 64), (200, 128), (321, 64), (520, 128)]


@pytest.mark.parametrize("form", ["4", "8", "8x2h", "t", "s1", "s3"])
@pytest.mark.parametrize("Sq,Skv,H,Hkv,D", [(1, 64, 2, 2, 64), (63, 63, 2, 2, 128), (65, 65, 2, 2, 64), (200, 200, 2, 2, 128), (321, 321, 2, 2, 64), (520, 520, 2, 2, 128),
                                           (130, 700, 4, 1, 128), (33, 321, 4, 2, 64)])
@pytest.mark.parametrize("cap", [33.3, 0.1, 1e4])
def test_soft_cap(monkeypatch, form, Sq, Skv, H, Hkv, D, cap):
  q, k, v = oracle.prepare_inputs(2, Sq, H, D, seed=Skv, kv_len=Skv)
  q, k, v = q * 2, k[:, :, :Hkv].contiguous(), v[:, :, :Hkv].contiguous()
  monkeypatch.setenv("FT_ATTN_FORM", form)
  out = ops.gemma2(q.cuda(), k.cuda(), v.cuda(), softcap=cap).float().cpu()
  ref = oracle.gemma2_forward(q, *(t.repeat_interleave(H // Hkv, 2) for t in (k, v)), softcap=cap).float()
  # probabilities and outputs are halves: two roundings of 2^-11 at most a value, and few logits, on a rounding boundary, move by a unit
  assert (out - ref).norm() <= 2e-3 * ref.norm(), ((out - ref).norm() / ref.norm()).item()


# A logit on a rounding boundary moves by one fp16 ulp, at most 2^-7 for logits below 16, and its probability by that share; outputs are
# means of values below 5 weighted by such probabilities, a few of which count: 5 * 2^-8, rounded up
O_BAR = 2e-2


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


def _capped(D, cap, singly=False):
  """Every positive finite half as a product of q and k, and its capped logit by the oracle's chain of halves, the last product an fp32
  number first (singly: rounded once, straight to a half), for those whose other roundings are no matter of a unit in the last places."""
  x = torch.arange(1, 0x7c00, dtype=torch.int16).view(torch.float16)
  t = x / math.sqrt(D)
  y = t / cap
  z = torch.tanh(y)
  c = torch.from_numpy((z.numpy().astype("f8") * float(np.float32(cap))).astype("f2")) if singly else z * cap
  ulp = lambda h: torch.from_numpy(np.spacing(h.numpy())).double()
  clear = ((t.double() / cap - y.double()).abs() < 0.47 * ulp(y)) & ((torch.tanh(y.double()) - z.double()).abs() < 0.47 * ulp(z))
  return x, c, clear


@pytest.mark.parametrize("form", ["4", "8", "t", "s1"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cap", [57.6, 44.8, 22.4])
def test_soft_cap_rounds_the_product_twice(monkeypatch, form, D, cap):
  """Heads of one query and two keys whose capped logits c and c - 1 the output shows as exp(-1), over logits from 8 on that a product
  rounded straight to a half would move by a unit, 2^-7 or more.  The bar is that of four half units of fp16: the two
  probabilities in front of the second product, the two outputs."""
  x, c, clear = _capped(D, cap)
  other = _capped(D, cap, singly=True)[1]
  pick = ((c != other) & clear & (c >= 8)).nonzero()[:, 0]
  plain = ((c == other) & clear).nonzero()[:, 0]
  beside = plain[(c[plain].double() - (c[pick].double()[:, None] - 1)).abs().argmin(1)]
  H, bar = len(pick), 4 * 2**-11
  assert H > 50
  q, k, v = (torch.zeros(1, s, H, D, dtype=torch.float16) for s in (1, 2, 2))
  q[..., 0] = 1
  k[0, 0, :, 0], k[0, 1, :, 0] = x[pick], x[beside]
  v[0, 0, :, 0] = v[0, 1, :, 1] = 1
  monkeypatch.setenv("FT_ATTN_FORM", form)
  out = ops.gemma2(q.cuda(), k.cuda(), v.cuda(), softcap=cap)[0, 0].double().cpu()
  ratio = out[:, 0].log() - out[:, 1].log()
  want = lambda to: to[pick].double() - c[beside].double()
  assert ((want(c) - want(other)).abs() > 3 * bar).all()
  assert ((ratio - want(c)).abs() <= bar).all(), (ratio - want(c)).abs().max().item()


@pytest.mark.parametrize("form", ["4", "8", "t"])
@pytest.mark.parametrize("Sq,Skv,D", [(1, 9, 128), (1, 9, 64), (40, 40, 128), (130, 161, 128), (70, 70, 64)])
def test_both_passes_of_keyformer_round_alike(monkeypatch, form, Sq, Skv, D):
  """A row's perturbed probabilities, of the column pass, sum to 1 under the normaliser that the attention pass made, to fp32 rounding (some
  2^-24 times exponents below 64) if both passes see the same logits; a rounding that only one of them had shows a hundred times over."""
  H, bar = 16, 1e-5
  q, k, v = oracle.prepare_inputs(1, Sq, H, D, seed=Skv, kv_len=Skv)
  q = q * 4
  er = oracle.prepare_exp_rand(1, H, Sq, Skv, seed=Skv)
  raw = torch.matmul(q.transpose(1, 2).double(), k.permute(0, 2, 3, 1).double())
  halves = (raw.half() / math.sqrt(D)).double()
  hidden = torch.ones(Sq, Skv).triu(Skv - Sq + 1).bool()
  z = lambda logits: (logits - er.double().log()).masked_fill(hidden, -math.inf)
  norm = z(halves).logsumexp(-1, keepdim=True)
  for other in (raw / math.sqrt(D), raw.half().double() / math.sqrt(D)) if D == 128 else (raw / math.sqrt(D),):  # a rounding left out
    assert ((z(other) - norm).exp().sum((2, 3)) / Sq - 1).abs().max() > 5 * bar
  monkeypatch.setenv("FT_ATTN_FORM", form)
  _, score = ops.keyformer(q.cuda(), k.cuda(), v.cuda(), er.cuda(), tau=1.0)
  total = score.double().sum(2).cpu() / Sq
  assert (total - 1).abs().max() <= bar, (total - 1).abs().max().item()


def test_soft_cap_waves_of_the_first_rows_hold_up_no_others():
  """Two tiles under the mask, of which the first 64 rows have one, take no longer than without it, where all rows have two (0.98 of the
  time; 1.08 where the barrier between the two tiles stood in the middle of the first one)."""
  q, k, v = (t.cuda() for t in oracle.prepare_inputs(1, 128, 8, 64, seed=5))
  graphs = []
  for causal in (True, False):
    ops.gemma2(q, k, v, softcap=50.0, causal=causal)
    torch.cuda.synchronize()
    graphs.append(torch.cuda.CUDAGraph())
    with torch.cuda.graph(graphs[-1]):
      for _ in range(50):
        ops.gemma2(q, k, v, softcap=50.0, causal=causal)
  least = [math.inf, math.inf]
  for _ in range(12):
    for i, g in enumerate(graphs):
      g.replay()
      begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
      begin.record()
      g.replay()
      end.record()
      end.synchronize()
      least[i] = min(least[i], begin.elapsed_time(end))
  assert least[0] <= 1.04 * least[1], least
