"""What this framework is timed on: the work that a program gives its operators, from a generation step of one query
row to the largest prompts and batches.

`listed()` names twelve cases, `draw(rng)` gives others of the same families and ranges, `prepare` makes what the program
has in hand before the call, `run` is one call through the public operators, `work` what it cannot do without and
`tolerance` how far another correct implementation at the same precision may be off.

Shapes: q [B, Sq, H, D], k and v [B, Skv, Hkv, D] for the softmax operators, q, k, v [B, S, H, D] for the linear ones
(here Sq = Skv = S), x [B, S, H * D] for the whole linear-attention function.
"""
import math

import torch

from flashtensor_amd import ops

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
GROUPED = ("attn", "h2o", "snapkv", "gemma2")  # operators that take fewer k/v heads than query heads
LINEAR = ("ea", "sima")
BLOCKS = ("ea_block", "sima_block")

# upper ends of the ranges: the largest listed cases
MOST_PAIRS = 4 * 32 * 4096 * 4096       # B H Sq Skv of a causal softmax call
MOST_BYTES = 1 << 30                    # tensors of a linear call, k and v of a generation step
MOST_GEMM = 8 * 8 * 8192 * 1024 * 1024  # 8 M C^2: the projections of a whole linear-attention function


def _softmax(name, op, B, H, Hkv, Sq, Skv, D, dtype="f16", causal=True, **more):
  return dict(name=name, op=op, B=B, H=H, Hkv=Hkv, Sq=Sq, Skv=Skv, D=D, dtype=dtype, causal=causal, **more)


def _linear(name, op, B, H, S, D, dtype, **more):
  return dict(name=name, op=op, B=B, H=H, Sq=S, D=D, dtype=dtype, **more)


def listed():
  return [
      # a short prompt: the call is its launch and the host path
      _softmax("attn_short", "attn", 1, 8, 8, 200, 200, 64),
      # a generation step of a small batch over the k/v cache, with its share of the heavy-hitter scores
      _softmax("h2o_generation", "h2o", 4, 32, 8, 1, 4097, 128, cached=True),
      # the scores a window of last queries gives the keys of a long prompt (SnapKV's observation window)
      _softmax("snapkv_window", "snapkv", 1, 32, 32, 64, 8000, 128, kernel_size=5),
      # one chunk of a prompt that is taken in pieces, grouped queries, soft-capped logits
      _softmax("gemma2_chunk", "gemma2", 1, 32, 8, 777, 3000, 128, "bf16", softcap=50.0),
      # prompts at the benchmark's configurations: scores and heavy hitters, the headline length, a batch
      _softmax("h2o_topk_prompt", "h2o", 1, 32, 32, 2048, 2048, 128, topk=256),
      _softmax("h2o_prompt", "h2o", 1, 32, 32, 4096, 4096, 128),
      _softmax("roco_batch", "roco", 4, 32, 32, 4096, 4096, 128),
      # KeyFormer with noise from a seed, and with the noise tensor its definition takes
      _softmax("keyformer_seeded", "keyformer", 1, 32, 32, 4096, 4096, 128, tau=1.0, noise="seed"),
      _softmax("keyformer_tensor", "keyformer", 1, 32, 32, 4096, 4096, 128, tau=1.5, noise="tensor"),
      # the linear core at its benchmark size
      _linear("ea_long", "ea", 8, 16, 8192, 64, "f16"),
      # the whole linear-attention function: its original shape and type, and a wide model over long sequences
      _linear("sima_block_narrow", "sima_block", 64, 4, 784, 32, "f32", normalize_q=False),
      _linear("ea_block_wide", "ea_block", 8, 16, 8192, 64, "f16"),
  ]


def _log_int(rng, lo, hi):
  return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_prompt(rng):
  op = rng.choice(("attn", "h2o", "h2o", "roco", "snapkv", "corm", "gemma2"))
  S, H = _log_int(rng, 64, 4096), rng.choice((8, 16, 32))
  B = _log_int(rng, 1, 8)
  causal = op not in ("attn", "h2o") or rng.random() < 0.85
  while B > 1 and B * H * S * S * (1 if causal else 2) > MOST_PAIRS:
    B -= 1
  dtype = rng.choice(("f16", "f16", "bf16"))
  c = _softmax("", op, B, H, H // 4 if op in GROUPED and rng.random() < 0.3 else H, S, S, rng.choice((64, 128, 128)), dtype, causal)
  if op == "h2o" and dtype == "f16" and rng.random() < 0.5:
    c["topk"] = max(1, S // 8)
  return c


def _draw_generation(rng):
  op = rng.choice(("attn", "h2o", "gemma2"))
  Sq = 1 if rng.random() < 0.6 else rng.randint(2, 8)  # one token, or a few proposed ones to be verified
  Skv, H, D = _log_int(rng, 256, 16384), rng.choice((16, 32)), rng.choice((64, 128, 128))
  Hkv = rng.choice((H // 4, H // 4, H))
  B = _log_int(rng, 1, 16)
  while B * Hkv * Skv * D * 4 > MOST_BYTES:
    B -= 1
  return _softmax("", op, B, H, Hkv, Sq, Skv, D, rng.choice(("f16", "f16", "bf16")), True, cached=True)


def _draw_chunk(rng):
  op = rng.choice(("attn", "h2o", "roco", "snapkv", "gemma2"))
  Sq, H = _log_int(rng, 16, 1024), rng.choice((8, 16, 32))
  Skv = _log_int(rng, max(1024, 2 * Sq), 16384)
  return _softmax("", op, 1, H, H // 4 if op in GROUPED and rng.random() < 0.5 else H, Sq, Skv, rng.choice((64, 128, 128)),
                  rng.choice(("f16", "f16", "bf16")))


def _draw_keyformer(rng):
  S, H = _log_int(rng, 200, 4096), rng.choice((8, 16, 32))
  return _softmax("", "keyformer", 1, H, H, S, S, rng.choice((64, 128, 128)), rng.choice(("f16", "f16", "f16", "bf16")),
                  tau=rng.choice((1.0, 1.0, 1.5, round(rng.uniform(0.5, 2.0), 2))), noise=rng.choice(("seed", "tensor")))


def _draw_linear(rng):
  dtype, D = rng.choice(("f16", "f16", "bf16", "f32")), rng.choice((64, 64, 64, 32))
  H, S, B = rng.choice((4, 8, 16)), _log_int(rng, 64, 16384), _log_int(rng, 1, 16)
  while 4 * B * S * H * D * (4 if dtype == "f32" else 2) > MOST_BYTES:
    B -= 1
  op = rng.choice(LINEAR)
  return _linear("", op, B, H, S, D, dtype, **({"normalize_q": rng.random() < 0.5} if op == "sima" else {}))


def _draw_block(rng):
  op = rng.choice(BLOCKS)
  if rng.random() < 0.5:  # narrow: heads of 32, two or four of them
    H, D, dtype = rng.choice((2, 4, 4)), 32, rng.choice(("f16", "bf16", "f32", "f32"))
  else:
    H, D, dtype = rng.choice((4, 8, 16)), 64, rng.choice(("f16", "f16", "bf16"))
  S, B = _log_int(rng, 64, 8192), _log_int(rng, 1, 64)
  while B > 1 and (8 * B * S * (H * D)**2 > MOST_GEMM or B * S > 1 << 16):
    B -= 1
  return _linear("", op, B, H, S, D, dtype, **({"normalize_q": rng.random() < 0.5} if op == "sima_block" else {}))


def draw(rng):
  c = rng.choice((_draw_prompt, _draw_prompt, _draw_generation, _draw_chunk, _draw_keyformer, _draw_linear, _draw_block))(rng)
  del c["name"]
  return c


def prepare(case, seed):
  """Inputs ~ N(0, 1) as in every case's own recipe; noise 1 + |N(0, 1)|; weights ~ N(0, 1 / C), biases 0.1 N(0, 1)."""
  dev = torch.device("cuda", torch.cuda.current_device())
  gen = torch.Generator(device=dev)
  gen.manual_seed(seed)
  dtype = DTYPES[case["dtype"]]
  B, H, D, Sq = case["B"], case["H"], case["D"], case["Sq"]

  def randn(*shape, t=dtype):
    return torch.randn(*shape, dtype=t, device=dev, generator=gen)

  s = {"case": case}
  if case["op"] in BLOCKS:
    C = H * D
    s["args"] = (randn(B, Sq, C), (randn(3 * C, C, t=torch.float32) / C**0.5).to(dtype), (0.1 * randn(3 * C, t=torch.float32)).to(dtype),
                 (randn(C, C, t=torch.float32) / C**0.5).to(dtype), (0.1 * randn(C, t=torch.float32)).to(dtype), H)
  elif case["op"] in LINEAR:
    s["args"] = tuple(randn(B, Sq, H, D) for _ in range(3))
  else:
    Skv, Hkv = case["Skv"], case["Hkv"]
    # a k/v cache has room for more tokens than it holds
    room = (Skv + 1023) // 1024 * 1024 if case.get("cached") else Skv
    s["args"] = (randn(B, Sq, H, D), randn(B, room, Hkv, D)[:, :Skv], randn(B, room, Hkv, D)[:, :Skv])
    if case.get("noise") == "tensor":
      s["exp_rand"] = randn(B, H, Sq, Skv, t=torch.float32).abs_().add_(1)
    s["seed"] = seed
  return s


def run(s):
  case, args = s["case"], s["args"]
  op = case["op"]
  if op == "attn":
    return ops.attn(*args, causal=case["causal"])
  if op == "h2o":
    out, score = ops.h2o(*args, causal=case["causal"])
    return (out, score, ops.topk(score, case["topk"])) if case.get("topk") else (out, score)
  if op == "roco":
    return ops.roco(*args)
  if op == "snapkv":
    return ops.snapkv(*args, kernel_size=case.get("kernel_size", 5))
  if op == "corm":
    return ops.corm(*args)
  if op == "gemma2":
    return ops.gemma2(*args, softcap=case.get("softcap", 50.0))
  if op == "keyformer":
    return ops.keyformer(*args, s.get("exp_rand"), tau=case["tau"], seed=s["seed"])
  if op == "ea":
    return ops.ea(*args)
  if op == "sima":
    return ops.sima(*args, normalize_q=case["normalize_q"])
  if op == "ea_block":
    return ops.ea_block(*args)
  return ops.sima_block(*args, normalize_q=case["normalize_q"])


def work(case):
  B, H, D, S = case["B"], case["H"], case["D"], case["Sq"]
  e = 4 if case["dtype"] == "f32" else 2
  if case["op"] in LINEAR:
    return {"bytes": 4 * B * S * H * D * e, "flops": 4 * B * H * S * D * D}
  if case["op"] in BLOCKS:
    C, M = H * D, B * S
    return {"bytes": (2 * M * C + 4 * C * C + 4 * C) * e, "flops": 8 * M * C * C + 4 * M * C * D}
  Hkv, Skv = case["Hkv"], case["Skv"]
  pairs = S * (Skv - S) + S * (S + 1) // 2 if case["causal"] else S * Skv
  nbytes = (2 * B * S * H * D + 2 * B * Skv * Hkv * D) * e  # q, out; k, v
  if case["op"] in ("h2o", "snapkv", "keyformer"):
    nbytes += B * Hkv * Skv * 4
  elif case["op"] == "roco":
    nbytes += 2 * B * H * Skv * 4
  elif case["op"] == "corm":
    nbytes += B * H * Skv
  if case.get("topk"):
    nbytes += B * Hkv * case["topk"] * 8
  if case.get("noise") == "tensor":
    nbytes += B * H * pairs * 4
  return {"bytes": nbytes, "flops": 4 * B * H * D * pairs}


def tolerance(case):
  # 16-bit operands and results; probabilities are rounded to the operand type in front of the second product, and a
  # logit whose exact value lies on a rounding boundary may go either way.  fp32 linear attention computes on fp16
  # operands.  Ranks and keep flags may differ where two scores, or a score and its threshold, meet.
  t = {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
  if case.get("topk"):
    t["differ"] = 1e-2
  elif case["op"] == "corm":
    t["differ"] = 1e-3
  return t
