"""Top-k at the lengths and counts where the kernel that ranks a row changes, against a stable sort: scores without a tie, with
many, all alike, and of every magnitude and sign (infinities too).  Whole numbers: no tolerance."""
import pytest
import torch

from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [512, 513, 1024, 1025, 1535, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193, 16385, 40000])
@pytest.mark.parametrize("scores", ["falling", "ties", "alike", "wide"])
def test_topk_at_the_edges_of_its_kernels(gpu, S, scores):
  g = torch.Generator().manual_seed(S)
  x = torch.rand(3, S, generator=g)
  if scores == "falling":
    x = x.cumsum(1).flip(1)
  elif scores == "ties":
    x = (x * 5).floor()
  elif scores == "alike":
    x = torch.full_like(x, 0.25)
  else:
    x = torch.randn(3, S, generator=g) * (60 * x - 30).exp()
    x[0, S // 2], x[1, S - 1], x[2, 0] = torch.inf, torch.inf, -torch.inf
  order = torch.sort(x, dim=-1, descending=True, stable=True).indices
  threads = max(64, 1 << (S - 1).bit_length() >> 3)
  for k in sorted({1, 2, S // 8, 128, 129, 256, 257, threads, threads + 1, 2 * threads, 2 * threads + 1, 4 * threads, 4 * threads + 1, S}):
    if k <= S and (S <= 8192 or k <= 16384):
      assert torch.equal(ops.topk(x.to(gpu), k).cpu(), order[:, :k]), k
