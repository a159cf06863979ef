"""Column sums of up to 64 rows from kept logits: row counts about the ends of a wave's rows and of the kernel's row counts (32, 48,
64), with groups, windows and sums of squares, against the CPU oracle.  Tolerances: half a unit of the 16-bit logits, relative,
in every probability (2e-3 fp16, 1e-2 bf16 of the norm), twice that for squares."""
import pytest
import torch

import oracle
from flashtensor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,H,Hkv", [(32, 4, 4), (33, 4, 4), (48, 4, 4), (49, 4, 4), (64, 4, 4), (65, 4, 4), (11, 6, 2), (16, 8, 2), (8, 8, 1)])
@pytest.mark.parametrize("Skv,D,dtype", [(200, 128, torch.float16), (449, 64, torch.float16), (1500, 128, torch.bfloat16)])
def test_sums_of_few_rows(gpu, Sq, H, Hkv, Skv, D, dtype):
  B, group, tol = 2, H // Hkv, 1e-2 if dtype is torch.bfloat16 else 2e-3
  q, k, v = oracle.prepare_inputs(B, Sq, H, D, seed=Sq + Skv, dtype=dtype, kv_len=Skv)
  k, v = k[:, :, :Hkv].contiguous(), v[:, :, :Hkv].contiguous()
  ref_o, ref_s, ref_sq = oracle.roco_forward(q, k.repeat_interleave(group, 2), v.repeat_interleave(group, 2))
  ref_s = ref_s.view(B, Hkv, group, Skv).mean(2)
  dev = [t.to(gpu) for t in (q, k, v)]

  def near(got, ref, t):
    got, ref = got.float().cpu(), ref.float()
    assert (got - ref).norm() <= t * ref.norm(), ((got - ref).norm() / ref.norm()).item()

  out, s = ops.h2o(*dev)
  near(out, ref_o, tol)
  near(s, ref_s, tol)
  for window in (3, 65):
    near(ops.snapkv(*dev, kernel_size=window)[1], torch.nn.functional.avg_pool1d(ref_s, window, 1, window // 2), tol)
  if group == 1:
    out, s, sq = ops.roco(*dev)
    near(out, ref_o, tol)
    near(s, ref_s, tol)
    near(sq, ref_sq, 2 * tol)
