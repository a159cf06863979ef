"""Sizes and counts beyond 32 bits are refused, not cut to their lower half: none of these calls queues a kernel."""
import pytest
import torch

from flashtensor_amd import ops

pytestmark = pytest.mark.gpu

WIDE = (2**31, 2**32 + 5, -2**32 + 5, 2**63, -2**64)


@pytest.mark.parametrize("n", WIDE)
def test_counts(gpu, n):
  q = torch.randn(1, 8, 2, 64, dtype=torch.float16, device=gpu)
  with pytest.raises(ValueError, match="32 bits"):
    ops.topk(torch.rand(2, 64, device=gpu), n)
  with pytest.raises(ValueError, match="32 bits"):
    ops.snapkv(q, q, q, kernel_size=n)
  x, w = torch.randn(1, 8, 64, dtype=torch.float16, device=gpu), torch.randn(192, 64, dtype=torch.float16, device=gpu)
  with pytest.raises(ValueError, match="32 bits"):
    ops.ea_block(x, w, None, w[:64], None, n)


def test_counts_at_the_edge_are_judged_as_before(gpu):
  """2^31 - 1 fits: refused for what it asks, not for its width."""
  with pytest.raises(ValueError, match="odd and positive"):
    ops.snapkv(*(torch.randn(1, 8, 2, 64, dtype=torch.float16, device=gpu),) * 3, kernel_size=-2**31)
  with pytest.raises(TypeError):
    ops.topk(torch.rand(2, 64, device=gpu), 3.5)


def test_sizes(gpu):
  """Lengths of 2^32 and a little, over storage that is nearly all shared or never written."""
  n = 2**32 + 64
  row = torch.empty(n, device=gpu)  # 17 GB
  with pytest.raises(ValueError, match="32 bits"):
    ops.topk(row, 8)
  del row
  q = torch.randn(1, 8, 2, 64, dtype=torch.float16, device=gpu)
  far = q[:, :1].expand(1, n, 2, 64)
  for op in (ops.attn, ops.h2o, ops.snapkv, ops.gemma2):
    with pytest.raises(ValueError, match="32 bits"):
      op(q, far, far)
  with pytest.raises(ValueError, match="32 bits"):
    ops.ea(far, far, far)
  with pytest.raises(ValueError, match="32 bits"):
    ops.attn(*(q[:, :1].expand(n, 1, 2, 64),) * 3)
  x, w = torch.randn(1, 1, 64, dtype=torch.float16, device=gpu), torch.randn(192, 64, dtype=torch.float16, device=gpu)
  with pytest.raises(ValueError):  # (an expanded x is not contiguous either)
    ops.ea_block(x.expand(1, n, 64), w, None, w[:64], None, 2)
