"""SnapKV's window over the column sums inside the column pass (widths up to 5) and in a launch of its own (wider ones): every form of the
pass, key counts around what a workgroup of 64 or 128 keys puts out, queries that see few or none of the first keys' rows,
grouped heads, against the window means of the sums themselves."""
import pytest
import torch

from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["1", "1t", "2"])
@pytest.mark.parametrize("Sq,Skv,H,Hkv,D,dtype,causal", [
    (1, 1, 2, 2, 64, torch.float16, True), (60, 60, 2, 2, 128, torch.float16, True), (61, 61, 2, 2, 64, torch.float16, True),
    (40, 124, 4, 1, 128, torch.bfloat16, True), (125, 125, 2, 2, 128, torch.float16, True), (300, 372, 4, 2, 128, torch.float16, True),
    (50, 241, 2, 2, 64, torch.float16, False), (513, 513, 4, 2, 64, torch.bfloat16, True)])
def test_windows(gpu, monkeypatch, form, Sq, Skv, H, Hkv, D, dtype, causal):
  monkeypatch.setenv("FT_ATTN_FORM", "4")  # the column pass whatever the number of rows
  monkeypatch.setenv("FT_COLSTATS_KEYS", form)
  g = torch.Generator().manual_seed(Skv)
  q, k, v = (torch.randn(2, s, h, D, dtype=dtype, generator=g).to(gpu) for s, h in ((Sq, H), (Skv, Hkv), (Skv, Hkv)))
  for fast in (False, True):
    sums = ops.h2o(q, k, v, causal=causal, fast_logits=fast)[1]
    for width in (1, 3, 5, 7):
      got = ops.snapkv(q, k, v, kernel_size=width, causal=causal, fast_logits=fast)[1]
      ref = torch.nn.functional.avg_pool1d(sums, width, 1, width // 2)
      # the same sums; up to seven of them added and divided, and the mean over a group's heads, in another order
      torch.testing.assert_close(got, ref, rtol=16 * 2**-24, atol=0)
