"""Torch-facing operators over the C ABI: one function per fused workload.

Call convention of the reference's emitted kernel wrapper (lib/Translate/to_triton.cpp:540-609): positional
torch tensors in, results allocated with torch.empty on the device of the first argument and returned
(a tuple when there are several), launch on the current stream, no synchronisation.  Torch is used for
device memory and the stream handle only; all arithmetic happens in libflashtensor_hip.  The checks, the
allocations and the call are native code (csrc/ops_torch.cpp, module ft_ops): bad arguments raise ValueError,
everything else RuntimeError, as std::invalid_argument / std::runtime_error do in the reference's ffi/ layer
(ffi/passes.cpp:81-83).  A tensor the kernels cannot read in place (a strided last axis) is refused, never copied.
"""
import torch

from . import _lib


_native = _lib.native


def attn(q, k, v, causal=True, fast_logits=False, return_lse=False):
  """Attn.forward (cases/kernels/attn.py:18-34): q [B,S,H,D], k,v [B,Skv,Hkv,D] -> out [B,Sq,H,D].  With
  Hkv < H query head h attends to k/v head h // (H // Hkv), the grouping of cases/attn.py:29-31."""
  return _native().attn(q, k, v, causal, fast_logits, return_lse)


def h2o(q, k, v, causal=True, fast_logits=False):
  """H2O.forward (cases/kernels/h2o.py:18-38) -> (out, h2o_score [B,Hkv,Skv] fp32); under grouped queries
  the probabilities are averaged over each group's query heads before the sum (cases/attn_h2o.py:42-47)."""
  return _native().h2o(q, k, v, causal, fast_logits)


def roco(q, k, v, causal=True, fast_logits=False):
  """RoCo.forward (cases/kernels/roco.py:18-48) -> (out, roco_score, roco_sq_score), scores [B,H,Skv] fp32."""
  return _native().roco(q, k, v, causal, fast_logits)


def keyformer(q, k, v, exp_rand=None, tau=1.5, seed=0, causal=True, fast_logits=False):
  """KeyFormer.forward (cases/kernels/kf.py:19-42) -> (out, kf_score [B,H,Skv] fp32).
  exp_rand [B,H,Sq,Skv] fp32 is the reference's noise input; None draws it in-kernel from `seed`."""
  return _native().keyformer(q, k, v, exp_rand, tau, int(seed), causal, fast_logits)


def snapkv(q, k, v, kernel_size=5, causal=True, fast_logits=False):
  """SnapKV.forward (cases/kernels/snapkv.py:19-43) -> (out, snapkv_score [B,H,Skv] fp32): the H2O column
  sums smoothed by a stride-1 average pool of odd width `kernel_size` over the key axis."""
  return _native().snapkv(q, k, v, int(kernel_size), causal, fast_logits)


def corm(q, k, v, corm_mask=None, causal=True, fast_logits=False, return_margin=False):
  """Corm.forward (cases/kernels/corm.py:18-40) -> (out, corm_score [B,H,Skv] bool): key j is kept when some
  query row gives it a probability >= corm_mask[i, j].  corm_mask [Sq,Skv] fp32 is the reference's input;
  None applies its prepare() recipe 1 / (i + 1) (corm.py:47-49) without reading a tensor."""
  return _native().corm(q, k, v, corm_mask, causal, fast_logits, return_margin)


def gemma2(q, k, v, softcap=50.0, causal=True, fast_logits=False):
  """Gemma2.forward (cases/kernels/gemma2.py:19-39): attention with logits softcap * tanh(logit / softcap)."""
  return _native().gemma2(q, k, v, softcap, causal, fast_logits)


def ea(q, k, v, out_dtype=None):
  """EA core (bench/ea.mlir:13-17): softmax(Q, dim=D) (softmax(K, dim=S)^T V); q,k,v [B,S,H,D] -> [B,S,H,D]."""
  return _native().linattn(q, k, v, _lib.FT_OP_EA, True, out_dtype)


def sima(q, k, v, normalize_q=True, out_dtype=None):
  """SimA core (bench/sima.mlir:13-17): L1-normalised Q, K over S per channel, O = Qh (Kh^T V).
  normalize_q=False multiplies by the raw Q as line 17 of the .mlir does."""
  return _native().linattn(q, k, v, _lib.FT_OP_SIMA, normalize_q, out_dtype)


def ea_block(x, w_qkv, b_qkv, w_out, b_out, head_num):
  """The whole function of bench/ea.mlir:2-23: q/k/v Linear, split into heads, EA core, output Linear.
  x [B,S,C], w_qkv [3C,C], b_qkv [3C], w_out [C,C], b_out [C] -> [B,S,C]."""
  return _native().linattn_block(x, w_qkv, b_qkv, w_out, b_out, head_num, _lib.FT_OP_EA, True)


def sima_block(x, w_qkv, b_qkv, w_out, b_out, head_num, normalize_q=True):
  """The whole function of bench/sima.mlir:2-23 (normalize_q as for `sima`)."""
  return _native().linattn_block(x, w_qkv, b_qkv, w_out, b_out, head_num, _lib.FT_OP_SIMA, normalize_q)


def topk(score, k):
  """Indices [..., k] (int64) of the k largest entries along the last axis, descending."""
  return _native().topk(score, k)


def seeded_exp_rand(B, H, Sq, Skv, seed, device):
  """The noise tensor the seeded KeyFormer mode draws, materialised on `device` ("cpu" uses the host twin)."""
  device = torch.device(device)
  out = torch.empty(B, H, Sq, Skv, dtype=torch.float32, device=device)
  seed = int(seed) & 0xFFFFFFFFFFFFFFFF
  if device.type == "cpu":
    _lib.ffi().kernels.noise_exp_fill_host(out.data_ptr(), B, H, Sq, Skv, seed)
  else:
    _lib.ffi().kernels.noise_exp_fill(out.data_ptr(), B, H, Sq, Skv, seed, torch.cuda.current_stream(device).cuda_stream)
  return out
