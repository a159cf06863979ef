"""The narrow linear-attention block over many token chunks: every workgroup of its output pass merges all of its batch's."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

# tokens to a chunk: 256, a strip of 32 for each of 8 waves, up to 64 chunks; the merge takes chunks by four up to 4 and by eight beyond


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,H", [(1, 1024, 4), (3, 1025, 4), (1, 2048, 2), (2, 2049, 4), (1, 16384, 2), (1, 16385, 4), (7, 7292, 4), (1, 33000, 2)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_block_over_many_chunks(B, S, H, dtype, monkeypatch):
  host = oracle.prepare_block_inputs(B, S, H, 32, seed=S % 97, dtype=dtype)
  dev = tuple(t.to("cuda") for t in host)
  last = (host[0][B - 1:],) + tuple(host[1:])
  # the result is a 16-bit tensor computed from 16-bit q, k, v and core: four roundings of 2^-9 (bf16: 2^-12 for fp16, whose operands
  # fp32 tensors take as well), each about a third of a unit in the mean
  bound = 4 * (2**-9 if dtype == torch.bfloat16 else 2**-12)
  for call, ref in ((lambda a: ops.ea_block(*a, H), lambda a: oracle.ea_block_forward(*a, H)),
                    (lambda a: ops.sima_block(*a, H), lambda a: oracle.sima_block_forward(*a, H)),
                    (lambda a: ops.sima_block(*a, H, normalize_q=False), lambda a: oracle.sima_block_forward(*a, H, normalize_q=False))):
    monkeypatch.delenv("FT_LINBLOCK_FORM", raising=False)
    y = call(dev)
    assert torch.equal(y, call(dev))  # one order of summation, whatever the workgroups' order
    monkeypatch.setenv("FT_LINBLOCK_FORM", "gemm")
    other = call(dev)
    for got in (y, other):
      assert torch.isfinite(got).all()
      want = ref(last).double()
      assert (got[B - 1:].double().cpu() - want).norm() <= bound * want.norm()
    assert (y.double() - other.double()).norm() <= 2 * bound * other.double().norm()
