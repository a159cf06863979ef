"""The forms of the attention pass that share out a row block's keys, between workgroups ("s") and between the two teams of
waves of one ("t"), against the CPU oracle: rows of one wave and of several, one off a block, shares of one tile or none,
keys one off a tile, rows that see no key of a share."""
import pytest
import torch

import oracle
from flashtensor_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["s1", "s3", "t"])
@pytest.mark.parametrize("Sq,Skv,H,Hkv,D,dtype", [
    (1, 65, 8, 2, 128, torch.float16), (1, 1000, 4, 4, 64, torch.bfloat16), (8, 449, 8, 2, 64, torch.float16), (33, 129, 4, 1, 128, torch.float16),
    (130, 1090, 4, 2, 64, torch.float16), (300, 300, 2, 2, 128, torch.float16), (257, 640, 2, 1, 128, torch.bfloat16),
    (1, 1, 1, 1, 128, torch.float16), (64, 64, 2, 2, 64, torch.bfloat16), (65, 65, 3, 3, 128, torch.float16), (63, 129, 2, 2, 64, torch.float16)])
def test_shares_of_the_keys(gpu, monkeypatch, form, Sq, Skv, H, Hkv, D, dtype):
  monkeypatch.setenv("FT_ATTN_FORM", form)
  g = torch.Generator().manual_seed(Sq + Skv)
  q, k, v = (torch.randn(s, h * D, dtype=dtype, generator=g) for s, h in ((Sq, H), (Skv, Hkv), (Skv, Hkv)))
  dev = [t.to(gpu).view(1, t.shape[0], -1, D) for t in (q, k, v)]
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  for causal in (True, False):
    ref_o, ref_s = oracle.attn_h2o2d_forward(q, k, v, Hkv, H, D, masked=causal)
    out, lse = ops.attn(*dev, causal=causal, return_lse=True)
    out2, score = ops.h2o(*dev, causal=causal)
    assert torch.isfinite(lse).all() and torch.equal(out, out2)
    ref = ref_o.float().view(1, Sq, H, D)
    assert (out.float().cpu() - ref).norm() <= tol * ref.norm()
    assert (score.cpu()[0] - ref_s).norm() <= tol * ref_s.norm()
  if H == Hkv:
    q4, k4, v4 = (t.view(1, t.shape[0], -1, D) for t in (q, k, v))
    ref = oracle.gemma2_forward(q4, k4, v4, 5.0).float()
    assert (ops.gemma2(*dev, softcap=5.0).float().cpu() - ref).norm() <= tol * ref.norm()


def test_a_workspace_without_room_for_the_shares_keeps_blocks_whole(gpu, monkeypatch):
  """The C ABI takes any workspace of at least ft_workspace_bytes(); only one of ft_workspace_bytes_split() lets it split."""
  monkeypatch.setenv("FT_ATTN_FORM", "s1")
  q, k, v = (torch.randn(1, s, 2, 64, dtype=torch.float16, device=gpu) for s in (4, 500, 500))
  k_ = _lib.ffi().kernels

  def args(o):
    return k_.AttnArgs(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), *(t.stride()[:3] for t in (q, k, v, o)), 1, 2, 4, 500, 64,
                       k_.F16, k_.CAUSAL, 2)

  a = args(torch.empty_like(q))
  need, more = (f(k_.OP_COLSTATS, a) for f in (k_.workspace_bytes, k_.workspace_bytes_split))
  assert more > need == 2 * 4 * 4
  ref = ops.h2o(q, k, v)
  for nbytes in (need, more - 1, more):
    out = torch.empty_like(q)
    score = torch.empty(1, 2, 500, device=gpu)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
    k_.attn_colstats_fwd(args(out), score.data_ptr(), 0, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    assert (out.float() - ref[0].float()).norm() <= 1e-3 * ref[0].float().norm() and torch.allclose(score, ref[1], rtol=1e-4)


@pytest.mark.parametrize("tiles", [0, 1])
@pytest.mark.parametrize("Sq,Skv,H,D,dtype", [(1, 2, 1, 128, torch.float16), (3, 447, 4, 64, torch.float16), (8, 448, 2, 128, torch.bfloat16),
                                              (17, 513, 2, 128, torch.float16), (32, 1025, 3, 64, torch.float16), (33, 600, 2, 64, torch.float16)])
def test_column_sums_of_few_rows(gpu, monkeypatch, tiles, Sq, Skv, H, D, dtype):
  """Up to 32 rows keep their logits for the column sums (key counts around the 448 and 512 keys of a workgroup, windows
  up to the widest that is taken in the same launch and one beyond), 33 go through the column pass."""
  if tiles:
    monkeypatch.setenv("FT_ATTN_FORM", f"s{tiles}")
  (q, k, v) = oracle.prepare_inputs(2, Sq, H, D, seed=Skv, dtype=dtype, kv_len=Skv)
  dev = [t.to(gpu) for t in (q, k, v)]
  tol = 1e-2 if dtype is torch.bfloat16 else 2e-3
  ref_o, ref_s, ref_sq = oracle.roco_forward(q, k, v)
  out, s, sq = ops.roco(*dev)
  assert (out.float().cpu() - ref_o.float()).norm() <= tol * ref_o.float().norm()
  assert (s.cpu() - ref_s).norm() <= tol * ref_s.norm() and (sq.cpu() - ref_sq).norm() <= 2 * tol * ref_sq.norm()
  for width in (1, 5, 65, 67):
    ref = torch.nn.functional.avg_pool1d(ref_s, width, 1, width // 2)
    assert (ops.snapkv(*dev, kernel_size=width)[1].cpu() - ref).norm() <= tol * ref.norm()


def _stored(t, layout):
  """The same values as views that programs hold: rows of a longer cache, heads of a packed tensor, [B, H, S, D] storage."""
  B, S, H, D = t.shape
  if layout == "cache":
    return torch.cat([t, t.new_full((B, 70, H, D), 9.0)], 1)[:, :S]
  if layout == "packed":
    return torch.cat([t.new_full((B, S, 1, D), 9.0), t, t.new_full((B, S, 2, D), 9.0)], 2)[:, :, 1:1 + H]
  return t.transpose(1, 2).contiguous().transpose(1, 2)


def _near(got, ref, tol):
  got, ref = got.float().cpu(), ref.float()
  assert (got - ref).norm() <= tol * ref.norm(), ((got - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("form", ["s1", "s3", "t", ""])
@pytest.mark.parametrize("layout", [("packed", "cache"), ("bhsd", "bhsd"), ("plain", "packed")])
@pytest.mark.parametrize("B,Sq,Skv,H,Hkv,D,dtype", [
    (3, 1, 321, 8, 2, 128, torch.float16), (2, 5, 450, 4, 1, 64, torch.bfloat16), (2, 40, 300, 6, 2, 64, torch.float16),
    (2, 33, 200, 3, 3, 128, torch.float16), (3, 2, 640, 2, 2, 64, torch.bfloat16), (2, 150, 513, 2, 2, 128, torch.float16)])
def test_shares_over_views_batches_and_groups(gpu, monkeypatch, form, layout, B, Sq, Skv, H, Hkv, D, dtype):
  monkeypatch.setenv("FT_ATTN_FORM", form)
  q, k, v = oracle.prepare_inputs(B, Sq, H, D, seed=Skv, dtype=dtype, kv_len=Skv)
  k, v = k[:, :, :Hkv].contiguous(), v[:, :, :Hkv].contiguous()
  dq, dk, dv = (t if lay == "plain" else _stored(t, lay) for t, lay in zip((q.to(gpu), k.to(gpu), v.to(gpu)), (layout[0], layout[1], layout[1])))
  group, tol = H // Hkv, 1e-2 if dtype is torch.bfloat16 else 2e-3
  kr, vr = (t.repeat_interleave(group, 2) for t in (k, v))  # query head h reads k/v head h // group
  ref_o, ref_s, ref_sq = oracle.roco_forward(q, kr, vr)
  ref_s = ref_s.view(B, Hkv, group, Skv).mean(2)
  out, lse = ops.attn(dq, dk, dv, return_lse=True)
  _near(out, ref_o, tol)
  logits = torch.matmul(q.transpose(1, 2).float(), kr.permute(0, 2, 3, 1).float()) / D**0.5
  logits += torch.full((Sq, Skv), -torch.inf).triu(Skv - Sq + 1)
  assert (lse.cpu() * 0.6931471805599453 - logits.logsumexp(-1)).abs().max() <= tol * logits.abs().where(logits.isfinite(), 0).max()
  out2, score = ops.h2o(dq, dk, dv)
  _near(out2, ref_o, tol)
  _near(score, ref_s, tol)
  _near(ops.gemma2(dq, dk, dv, softcap=5.0), oracle.gemma2_forward(q, kr, vr, 5.0), tol)
  _near(ops.snapkv(dq, dk, dv, kernel_size=7)[1], torch.nn.functional.avg_pool1d(ref_s, 7, 1, 3), tol)
  # logits kept in fp32: against the fp32 definition
  probs = logits.softmax(-1)
  fast_o = torch.matmul(probs.to(dtype).float(), vr.transpose(1, 2).float()).transpose(1, 2)
  out3, score3 = ops.h2o(dq, dk, dv, fast_logits=True)
  _near(out3, fast_o, tol)
  _near(ops.attn(dq, dk, dv, fast_logits=True), fast_o, tol)
  _near(score3, probs.sum(2).view(B, Hkv, group, Skv).mean(2), tol)
  if group == 1:
    out4, s1, s2 = ops.roco(dq, dk, dv)
    _near(out4, ref_o, tol)
    _near(s1, ref_s, tol)
    _near(s2, ref_sq, 2 * tol)
    out5, keep = ops.corm(dq, dk, dv)
    _near(out5, ref_o, tol)
    ratio = oracle.corm_margin(q, k, oracle.corm_mask_rule(Sq, Skv))  # a key is kept from 1 on; nearer than tol either way goes
    sure = (ratio - 1).abs() > tol
    assert torch.equal(keep.cpu()[sure], (ratio >= 1)[sure]) and sure.float().mean() > 0.9
  # no mask: every row sees every key of every share
  full_o, full_s = zip(*(oracle.attn_h2o2d_forward(*(t[b].reshape(t.shape[1], -1) for t in (q, k, v)), Hkv, H, D, masked=False) for b in range(B)))
  out6, score6 = ops.h2o(dq, dk, dv, causal=False)
  _near(out6, torch.stack(full_o).view(B, Sq, H, D), tol)
  _near(score6, torch.stack(full_s), tol)


def test_undivided_attention_allocates_its_result_only(gpu):
  """Plain attention over a chunk that only the soft-capped form divides."""
  q, k, v = (torch.randn(1, s, h, 128, dtype=torch.bfloat16, device=gpu) for s, h in ((777, 32), (3000, 8), (3000, 8)))
  for op, room in ((ops.attn, 0), (ops.gemma2, 50 << 20)):
    op(q, k, v)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = op(q, k, v)
    extra = torch.cuda.max_memory_allocated() - before - out.numel() * 2
    assert room <= extra < room + (20 << 20), extra
