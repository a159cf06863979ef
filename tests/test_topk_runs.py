"""Top-k by runs of one wave each: row lengths around the padded sizes, k at the length of a run and one beyond (which the
whole-row network takes), distinct scores and heavy ties, against a stable descending sort."""
import pytest
import torch

from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,run", [(500, 64), (512, 64), (513, 128), (1025, 256), (2048, 256), (2049, 512), (4096, 512), (4097, 1024), (8192, 1024)])
def test_k_around_the_length_of_a_run(gpu, S, run):
  g = torch.Generator().manual_seed(S)
  for score in (torch.randn(3, S, generator=g), torch.randint(0, 5, (3, S), generator=g).float()):
    want = torch.sort(score, dim=-1, descending=True, stable=True).indices
    for k in (1, run // 2, run // 2 + 1, run - 1, run, run + 1):
      assert torch.equal(ops.topk(score.to(gpu), k).cpu(), want[:, :k]), k
