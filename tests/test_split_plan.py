"""How attention divides its keys is decided on the host in front of every launch: the decision is cheap for shapes that are
new in every call (a generation loop's Skv grows by one a step), and the same for all of them with the same key tiles."""
import ctypes
import time

import pytest

from flashtensor_amd import _lib
from flashtensor_amd._lib import FtAttnArgs, FtStrides


def _args(B, H, Hkv, Sq, Skv, D, flags=_lib.FT_CAUSAL):
  st, sq = FtStrides(Skv * Hkv * D, Hkv * D, D), FtStrides(Sq * H * D, H * D, D)
  return FtAttnArgs(q=0x1000, k=0x2000, v=0x3000, o=0x4000, sq=sq, sk=st, sv=st, so=sq, B=B, H=H, Hkv=Hkv, Sq=Sq, Skv=Skv, D=D,
                    dtype=_lib.FT_F16, flags=flags)


def _bytes(op, *shape):
  return _lib.load().ft_workspace_bytes_split(op, ctypes.byref(_args(*shape)))


@pytest.mark.parametrize("op", [_lib.FT_OP_ATTN, _lib.FT_OP_COLSTATS])
@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,D", [(4, 32, 8, 1, 4097, 128), (16, 32, 8, 1, 16384, 64), (8, 32, 32, 1, 8192, 128),
                                              (16, 32, 32, 1, 8192, 64), (1, 32, 32, 64, 8000, 128), (2, 32, 32, 500, 9000, 128)])
def test_new_shapes_are_planned_in_microseconds(op, B, H, Hkv, Sq, Skv, D):
  """A search that simulates a launch for every number of shares takes 10 to 300 us a shape here."""
  f = _lib.load().ft_workspace_bytes_split
  best = float("inf")
  for rep in range(60):  # the quietest of many short spells: other processes may be busy
    args = [ctypes.byref(_args(B, H, Hkv, Sq, Skv + 64 * (i + 10 * rep), D)) for i in range(10)]
    t = time.thread_time()
    for a in args:
      f(op, a)
    best = min(best, (time.thread_time() - t) / len(args))
  assert best < 8e-6, f"{best * 1e6:.1f} us a shape"


@pytest.mark.parametrize("op", [_lib.FT_OP_ATTN, _lib.FT_OP_COLSTATS, _lib.FT_OP_SNAPKV])
@pytest.mark.parametrize("B,H,Hkv,Sq,D", [(4, 32, 8, 1, 128), (1, 32, 32, 64, 128), (2, 16, 4, 32, 64), (1, 8, 8, 128, 64)])
def test_one_plan_for_all_lengths_of_as_many_tiles(op, B, H, Hkv, Sq, D):
  need = _lib.load().ft_workspace_bytes
  pad = lambda n: -(-n // 256) * 256
  parts = {_bytes(op, B, H, Hkv, Sq, Skv, D) - pad(need(op, ctypes.byref(_args(B, H, Hkv, Sq, Skv, D)))) for Skv in range(64 * 63 + 1, 64 * 64 + 1, 7)}
  assert len(parts) == 1 and parts.pop() > 0


def test_each_form_of_attention_asks_for_its_own_workspace():
  """A chunk that only the soft-capped form divides (61 MB): the plain one needs nothing."""
  lib = _lib.load()
  a = _args(1, 32, 8, 777, 3000, 128)
  plain, capped = (lib.ft_attn_workspace_bytes(ctypes.byref(a), cap) for cap in (0.0, 50.0))
  assert plain == 0 and capped > 50 << 20 and lib.ft_workspace_bytes_split(_lib.FT_OP_ATTN, ctypes.byref(a)) == capped
  assert lib.ft_attn_workspace_bytes(ctypes.byref(_args(4, 32, 8, 1, 4097, 128)), 0.0) > 0
  for bad in (_args(1, 32, 5, 777, 3000, 128), _args(1, 32, 8, 0, 3000, 128), _args(0, 32, 8, 1, 3000, 128)):
    assert lib.ft_attn_workspace_bytes(ctypes.byref(bad), 0.0) == 0
  assert lib.ft_attn_workspace_bytes(None, 0.0) == 0
