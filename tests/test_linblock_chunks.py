"""The narrow linear-attention block over many token chunks: every workgroup of its output pass merges all of its batch's."""
import ctypes

import pytest
import torch

import oracle
from flashtensor_amd import _lib, ops

# Tokens to a chunk: 256, a strip of 32 for each of 8 waves, or as many strips more as 64 chunks or a round of 256 CUs make it.  The merge
# takes chunks by four, with four heads and more than four chunks by eight; with up to four one wave a head merges, of two heads in
# fp32 four.  The last column is the chunks of fp32 tensors, 0 where they leave the call to the library's products.
SHAPES = [(1, 20, 2, 1, 1), (1, 257, 2, 3, 3), (3, 128, 2, 4, 4), (1, 1024, 4, 4, 4), (3, 1025, 4, 5, 5), (1, 2048, 2, 8, 8), (2, 2049, 4, 9, 0), (30, 2049, 4, 8, 8),
          (28, 2296, 4, 9, 9), (16, 4096, 4, 16, 16), (17, 3841, 2, 14, 14), (1, 16384, 2, 64, 0), (1, 16385, 4, 57, 0), (7, 7292, 4, 29, 0), (1, 33000, 2, 61, 0)]
CASES = [(t, *s[:3], s[4] if t is torch.float32 else s[3]) for t in (torch.float16, torch.bfloat16, torch.float32) for s in SHAPES if t is not torch.float32 or s[4]]


def _chunks(B, S, H, dtype):
  plan = _lib.load()._ZN2ft16small_block_planERK14FtLinBlockArgsPiS3_  # ft::small_block_plan
  n, strips = ctypes.c_int(), ctypes.c_int()
  code = {torch.float16: _lib.FT_F16, torch.bfloat16: _lib.FT_BF16, torch.float32: _lib.FT_F32}[dtype]
  plan(ctypes.byref(_lib.FtLinBlockArgs(B=B, S=S, H=H, D=32, dtype=code)), ctypes.byref(n), ctypes.byref(strips))
  assert n.value == 0 or (n.value - 1) * strips.value < -(-S // 32) <= n.value * strips.value
  return n.value


@pytest.mark.parametrize("B,S,H,chunks,chunks32", SHAPES)
def test_chunks_of_a_call(B, S, H, chunks, chunks32):
  assert (_chunks(B, S, H, torch.float16), _chunks(B, S, H, torch.bfloat16), _chunks(B, S, H, torch.float32)) == (chunks, chunks, chunks32)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,B,S,H,chunks", CASES)
def test_block_over_many_chunks(dtype, B, S, H, chunks, monkeypatch):
  assert _chunks(B, S, H, dtype) == chunks  # the two launches, not the library's products
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
