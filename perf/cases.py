"""The work that users of this package have it do, as timed cases.

A case is a dict of plain values.  Its `kind` says which public entry point it calls:

  attn    recml_amd.hstu_attention / hstu_attention_autograd: padded or jagged batches, bias tables, dropout
  splash  recml_amd.pointwise_splash_attention, the reference-named operator: segment ids, window, full or causal
  dense   recml_amd.pointwise_attention, the layer-side call with a [B, L, L] mask and an additive bias
  model   recml_amd.HSTU: embedding, blocks, final norm and, where there is one, the output head

and `grad` whether the gradients are taken too (a training step's forward and backward).  Sizes are those of
recml_amd.workloads and bench.py, of the reference's operator test (B=128, L=512, H=8, d=128 in fp32) and of its
example model (50 positions, width 64, 4 heads, 4 layers); `draw` spreads the same kinds over their range.

The lengths of a batch come from the case alone (`len_seed`), so that its work is known without its inputs; which
sequence has which length, and every value, comes from the seed.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import recml_amd

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp8": torch.bfloat16}   # (fp8: q and k only)
_BYTES = {"fp32": 4, "bf16": 2, "fp8": 2}


def _attn(name, B, L, H, d, dtype, *, layout="padded", lens="full", pos=False, ts=False, dropout=0.0, grad=False, len_seed=1):
  return dict(name=name, kind="attn", B=B, L=L, H=H, d=d, dtype=dtype, layout=layout, lens=lens, pos=pos, ts=ts,
              dropout=dropout, grad=grad, len_seed=len_seed)


def _splash(name, B, L, H, d, dtype, *, causal=True, segments=False, window=0, grad=False, len_seed=1):
  return dict(name=name, kind="splash", B=B, L=L, H=H, d=d, dtype=dtype, causal=causal, segments=segments, window=window,
              lens="uniform", grad=grad, len_seed=len_seed)


def _dense(name, B, L, H, d, dtype, *, lens="full", bias=True, grad=False, len_seed=1):
  return dict(name=name, kind="dense", B=B, L=L, H=H, d=d, dtype=dtype, lens=lens, bias=bias, grad=grad, len_seed=len_seed)


def _model(name, B, L, H, d, layers, vocab, dtype, *, lens="uniform", pos=False, ts=False, head=False, jagged=True, grad=False,
           len_seed=1):
  return dict(name=name, kind="model", B=B, L=L, H=H, d=d, layers=layers, vocab=vocab, dtype=dtype, lens=lens, pos=pos, ts=ts,
              head=head, jagged=jagged, grad=grad, len_seed=len_seed)


def listed():
  return [
      # a unit-test sized call, Keras' default dtype: nothing but launches and host work
      _attn("tiny fp32 call", 4, 64, 2, 32, "fp32"),
      # a small padded batch of a ranking model's attention
      _attn("small padded bf16 call", 32, 512, 4, 64, "bf16", lens="uniform", pos=True, len_seed=2),
      # the headline batch: user histories of power-law length, packed, both bias tables
      _attn("jagged bf16 call", 64, 2048, 8, 128, "bf16", layout="jagged", lens="power", pos=True, ts=True, len_seed=3),
      # inference on long histories with 8-bit queries and keys
      _attn("long jagged fp8 call", 32, 4096, 8, 128, "fp8", layout="jagged", lens="uniform", pos=True, len_seed=5),
      # the headline batch in training
      _attn("jagged bf16 training", 64, 2048, 8, 128, "bf16", layout="jagged", lens="power", pos=True, ts=True, grad=True, len_seed=3),
      # training on full-length histories: the largest
      _attn("full-length bf16 training", 64, 2048, 8, 128, "bf16", layout="jagged", lens="full", pos=True, ts=True, grad=True),
      # the reference operator's own recipe: fp32, segment ids, out and gradients
      _splash("reference-named op fp32 training", 128, 512, 8, 128, "fp32", segments=True, grad=True, len_seed=7),
      # the layer-side call in inference
      _dense("dense mask and bias bf16 call", 16, 2048, 8, 128, "bf16"),
      # the layer-side call in training, the bias a trainable module's output, at a length that is no power of two
      _dense("dense mask and bias bf16 training", 16, 1000, 8, 64, "bf16", lens="uniform", grad=True, len_seed=8),
      # the example model scoring a small batch of requests
      _model("example model, scoring", 32, 50, 4, 16, 4, 20000, "bf16", head=True, jagged=False, len_seed=9),
      # the ranking model, inference on packed tokens
      _model("ranking model, inference", 128, 1024, 8, 64, 4, 1000000, "bf16", pos=True, len_seed=4),
      # the ranking model, forward and backward of a training step on packed tokens
      _model("ranking model, training", 128, 1024, 8, 64, 4, 100000, "bf16", pos=True, grad=True, len_seed=4),
  ]


def _log_int(rng, lo, hi):
  return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.99)))))))


def _cost(case):
  """What a drawn case may cost, in the units of the listed ones: bytes or flops, whichever is more at 50 flops a byte."""
  w = work(case)
  return max(w["bytes"], w["flops"] / 50)


def draw(rng):
  """One more case of the listed kinds.  Costs are capped by the listed case of the same kind and precision."""
  while True:
    kind = rng.choice(("attn", "attn", "attn", "splash", "dense", "model"))
    grad = rng.random() < 0.5
    B, L, H = _log_int(rng, 1, 192), _log_int(rng, 24, 4096), rng.choice((1, 2, 3, 4, 8, 8, 12, 16))
    d = rng.choice((32, 64, 128))
    dtype = rng.choice(("bf16", "bf16", "fp32"))
    len_seed = rng.randrange(1 << 16)
    if kind == "attn":
      pos = rng.random() < 0.7
      if dtype == "bf16" and not grad and rng.random() < 0.3:
        dtype = "fp8"
      case = _attn("", B, L, H, d, dtype, layout=rng.choice(("padded", "jagged")), lens=rng.choice(("uniform", "power", "full")),
                   pos=pos, ts=pos and rng.random() < 0.5, dropout=0.2 if grad and rng.random() < 0.25 else 0.0, grad=grad,
                   len_seed=len_seed)
    elif kind == "splash":
      case = _splash("", B, L, H, d, dtype, causal=rng.random() < 0.7, segments=rng.random() < 0.5,
                     window=rng.choice((0, 0, max(1, L // 4))), grad=grad, len_seed=len_seed)
    elif kind == "dense":
      case = _dense("", min(B, 64), min(L, 2048), H, d, dtype, lens=rng.choice(("uniform", "full")), bias=rng.random() < 0.6,
                    grad=grad, len_seed=len_seed)
    else:
      L = min(L, 1024)
      H, d = rng.choice((1, 2, 4, 8)), rng.choice((16, 32, 64, 128))
      head = rng.random() < 0.3
      case = _model("", B, L, H, d, rng.randint(2, 6), _log_int(rng, 1000, 20000 if head else 200000), dtype, pos=rng.random() < 0.7,
                    ts=rng.random() < 0.3, head=head, jagged=rng.random() < 0.6, grad=grad, len_seed=len_seed)
    del case["name"]
    slow = dtype == "fp32" or d not in (32, 64, 128)     # (general kernels: capped by the fp32 case)
    cap = "reference-named op fp32 training" if slow else {
        "attn": "full-length bf16 training", "splash": "full-length bf16 training", "dense": "dense mask and bias bf16 call",
        "model": "ranking model, training"}[kind]
    if _cost(case) <= next(_cost(c) for c in listed() if c["name"] == cap):
      return case


# ---------------------------------------------------------------------------
# lengths and work
# ---------------------------------------------------------------------------


def _lengths(case):
  """The batch's lengths before they are dealt to its sequences: full; U{L/8 .. L}; or a power law (exponent 1.2) from 16."""
  B, L = case["B"], case["L"]
  rng = np.random.default_rng(case["len_seed"])
  if case["lens"] == "uniform":
    return rng.integers(max(1, L // 8), L + 1, B).astype(np.int64)
  if case["lens"] == "power":
    lo, e = min(16, L), -0.2
    x = (lo**e + rng.random(B) * (L**e - lo**e)) ** (1.0 / e)
    return np.clip(np.floor(x), lo, L).astype(np.int64)
  return np.full(B, L, dtype=np.int64)


def _segments(case):
  """Splash batches with segment ids: how many positions of a row each of its two packed sequences takes (the rest is padding)."""
  n = _lengths(case)
  return n - n // 3, n // 3


def _pairs_of(n, causal, window):
  """(query, key) pairs kept in a run of n positions."""
  n = np.asarray(n, dtype=np.int64)
  w = np.minimum(n - 1, window) if window else n - 1
  w = np.maximum(w, 0)
  below = w * (w + 1) // 2 + (n - w - 1).clip(0) * w      # pairs with 0 < i - j <= w
  return int((below * (1 if causal else 2) + n).sum())


def _pairs(case):
  if case["kind"] == "splash":
    if case["segments"]:
      a, b = _segments(case)
      pad = case["L"] - a - b
      return sum(_pairs_of(x[x > 0], case["causal"], case["window"]) for x in (a, b, pad))
    return _pairs_of(np.full(case["B"], case["L"]), case["causal"], case["window"])
  return _pairs_of(_lengths(case), True, 0)


def work(case):
  B, L, H, d, grad = case["B"], case["L"], case["H"], case["d"], case["grad"]
  e = _BYTES[case["dtype"]]
  lens = _lengths(case)
  valid = int(lens.sum())
  pair_flops = (12 if grad else 4) * d * H * _pairs(case)     # two products forward, four more backward
  if case["kind"] == "model":
    D, n = H * d, case["layers"]
    T = valid if case["jagged"] else B * L
    width = case["vocab"] if case["head"] else D
    params = n * (5 * D * D + 4 * D) + 2 * D + L * D + (D * case["vocab"] if case["head"] else 0)
    flops = (3 if grad else 1) * (2 * T * 5 * D * D * n + (2 * T * D * width if case["head"] else 0)) + n * pair_flops
    rows = T * D * e                                           # the embedding rows that are read
    nbytes = T * 8 + rows + params * e + B * L * width * e
    if grad:
      nbytes += (params + case["vocab"] * D) * e + B * L * width * e
    return {"bytes": nbytes, "flops": flops}
  tokens = valid if case.get("layout") == "jagged" else B * L  # (output rows past a length are written as zeros)
  reads = B * L if case["kind"] == "splash" else valid
  qk = 1 if case["dtype"] == "fp8" else e
  nbytes = reads * H * d * (2 * qk + e) + tokens * H * d * e   # q, k, v in; out
  if grad:
    nbytes += reads * H * d * e + 3 * tokens * H * d * e       # dout in; dq, dk, dv out
  if case.get("pos"):
    nbytes += H * (2 * L - 1) * 4 * (2 if grad else 1)
  if case.get("ts"):
    nbytes += tokens * 8 + H * 129 * 4 * (2 if grad else 1)
  if case["kind"] == "dense":
    nbytes += B * L * L
    if case["bias"]:
      nbytes += B * L * L * 4 * (2 if grad else 1)
  return {"bytes": nbytes, "flops": pair_flops}


def tolerance(case):
  """fp32: sums in 32 bits.  bf16 (and fp8 operands, which are exact in it): the activated weights, the outputs and the gradients are
  each rounded to 8 bits once or twice; a model rounds at every step of every block."""
  if case["dtype"] == "fp32":
    return {"rel": 3e-5 if case["kind"] == "model" else 1e-5, "max": 2e-3}
  return {"rel": 2e-2 if case["kind"] == "model" else 1e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


class _Draws:
  """Device-side random values of one seed."""

  def __init__(self, seed):
    self.dev = torch.device("cuda")
    self.gen = torch.Generator(device=self.dev).manual_seed(seed)
    self.host = np.random.default_rng(seed)

  def normal(self, shape, std, dtype=torch.float32):
    return torch.randn(shape, device=self.dev, generator=self.gen).mul_(std).to(dtype)

  def uniform(self, shape):
    return torch.rand(shape, device=self.dev, generator=self.gen)

  def put(self, a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)


def _timestamps(r, B, L):
  """Seconds, an item about every hour: [B, L] int64, rising along every row."""
  gaps = torch.ceil(-torch.log1p(-r.uniform((B, L)).double()) * 3600.0).to(torch.int64)
  return 1_600_000_000 + torch.cumsum(gaps, 1)


def _to_fp8(x):
  """Per-head scales amax / 448 and e4m3 values."""
  xf = x.float()
  scale = xf.abs().amax(dim=tuple(i for i in range(x.dim()) if i != x.dim() - 2)) / 448.0
  return (xf / scale[:, None]).to(torch.float8_e4m3fn), scale.contiguous()


def _prepare_attention(case, r):
  B, L, H, d, grad, kind = case["B"], case["L"], case["H"], case["d"], case["grad"], case["kind"]
  dt = _DTYPES[case["dtype"]]
  lens = r.host.permutation(_lengths(case)).astype(np.int32)
  jagged = case.get("layout") == "jagged"
  shape = (int(lens.sum()), H, d) if jagged else (B, L, H, d)
  # the reference's operator test draws N(0, 1) and scales by 1/sqrt(d); the layer's projections are smaller
  std = 1.0 if kind == "splash" else 0.1
  q, k, v = (r.normal(shape, std, dt) for _ in range(3))
  kw, wrt = {}, []
  if kind == "attn":
    if jagged:
      kw.update(seq_offsets=r.put(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)), max_len=L)
    elif case["lens"] != "full":
      kw["seq_lens"] = r.put(lens)
    if case["dropout"] > 0:
      kw.update(dropout_p=case["dropout"], dropout_seed=int(r.host.integers(1 << 40)))
    if case["pos"]:
      kw["pos_bias"] = r.normal((H, 2 * L - 1), 0.02)
      wrt.append(kw["pos_bias"])
    if case["ts"]:
      ts = _timestamps(r, B, L)
      if jagged:
        ts = ts[torch.arange(L, device=r.dev)[None, :] < r.put(lens)[:, None]]
      kw.update(timestamps=ts, ts_bias=r.normal((H, 129), 0.02))
      wrt.append(kw["ts_bias"])
    if case["dtype"] == "fp8":
      q, kw["q_scale"] = _to_fp8(q)
      k, kw["k_scale"] = _to_fp8(k)
  elif kind == "splash":
    if case["segments"]:
      # two sequences packed into each row, then padding: ids 1, 2, 0
      order = r.host.permutation(B)
      a, b = (r.put(x[order]) for x in _segments(case))
      i = torch.arange(L, device=r.dev)[None, :]
      ids = torch.where(i < a[:, None], 1, torch.where(i < (a + b)[:, None], 2, 0)).to(torch.int32)
      kw.update(q_segment_ids=ids, kv_segment_ids=ids)
    if case["window"]:
      kw["sliding_window_size"] = case["window"]
  else:
    valid = torch.arange(L, device=r.dev)[None, :] < r.put(lens)[:, None]
    kw["attention_mask"] = recml_amd.make_causal_mask(valid, dtype=torch.bool)
    kw["attention_bias"] = r.normal((B, L, L), 0.02) if case["bias"] else None
    if case["bias"]:
      wrt.append(kw["attention_bias"])
  state = dict(kind=kind, grad=grad, q=q, k=k, v=v, kw=kw, causal=case.get("causal", True))
  if grad:
    state["wrt"] = [q, k, v] + wrt
    for t in state["wrt"]:
      t.requires_grad_(True)
    state["dout"] = r.normal(shape, 1.0, dt)
  return state


def _prepare_model(case, r, seed):
  B, L, H, d, grad = case["B"], case["L"], case["H"], case["d"], case["grad"]
  dt, D = _DTYPES[case["dtype"]], H * d
  model = recml_amd.HSTU(vocab_size=8, max_positions=L, model_dim=D, num_heads=H, num_layers=case["layers"], add_head=False, dtype=dt,
                         device=r.dev, seed=seed)
  P = torch.nn.Parameter
  model.item_embedding = P(r.normal((case["vocab"], D), 0.02, dt), requires_grad=False)
  if case["head"]:
    model.reverse_embedding = P(r.normal((D, case["vocab"]), 0.02, dt), requires_grad=False)
  lens = r.put(r.host.permutation(_lengths(case)).astype(np.int32))
  valid = torch.arange(L, device=r.dev)[None, :] < lens[:, None]
  # popular items come up far more often than others (log-uniform ranks); 0 pads
  ids = torch.exp(r.uniform((B, L)).double() * math.log(case["vocab"])).to(torch.int64).clamp_(1, case["vocab"] - 1) * valid
  kw = dict(seq_lens=lens, jagged=True) if case["jagged"] else dict(padding_mask=valid)
  wrt = []
  if case["pos"]:
    kw["pos_bias"] = r.normal((2 * L - 1,), 0.02)
    wrt.append(kw["pos_bias"])
  if case["ts"]:
    kw.update(timestamps=_timestamps(r, B, L), ts_bias=r.normal((129,), 0.02))
    wrt.append(kw["ts_bias"])
  state = dict(kind="model", grad=grad, model=model, ids=ids, kw=kw)
  if grad:
    model.requires_grad_(True)
    for t in wrt:
      t.requires_grad_(True)
    state["wrt"] = list(model.parameters()) + wrt
    state["dout"] = r.normal((B, L, case["vocab"] if case["head"] else D), 1.0, dt)
  return state


def prepare(case, seed):
  r = _Draws(seed)
  return _prepare_model(case, r, seed) if case["kind"] == "model" else _prepare_attention(case, r)


def _forward(s):
  if s["kind"] == "model":
    return s["model"](s["ids"], **s["kw"])
  if s["kind"] == "splash":
    kind = recml_amd.MaskType.CAUSAL if s["causal"] else recml_amd.MaskType.FULL
    return recml_amd.pointwise_splash_attention(kind, s["q"], s["k"], s["v"], **s["kw"])
  if s["kind"] == "dense":
    return recml_amd.pointwise_attention(s["q"], s["k"], s["v"], **s["kw"])
  op = recml_amd.hstu_attention_autograd if s["grad"] else recml_amd.hstu_attention
  return op(s["q"], s["k"], s["v"], **s["kw"])


def run(state):
  if not state["grad"]:
    with torch.no_grad():
      return _forward(state)
  out = _forward(state)
  return [out.detach(), *torch.autograd.grad(out, state["wrt"], state["dout"])]
