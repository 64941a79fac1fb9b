"""What a user of this runtime has it do, as cases that can be timed and checked: decode steps, prompts, generation and
training steps through ShardRunner and ShardTrainer, on the shards that ring peers hold.

Every model here has its real layer sizes (models.config presets; the mixed-layer designs at the sizes bench.py gives
them), random weights and, where a whole model would not be needed to see its cost, the layers of a ring's last peer, LM
head included: such a peer receives hidden states.  Decode steps and prompts of stateless models run on requests that are
rolled back after the pass, so a pass can be repeated; models with recurrent state serve their requests from admission to
the end.  Tokens are given, as when recorded traffic is replayed; outputs are logits.

exact() is the same arithmetic in float64 from plain torch, whole sequences at once.
"""
import itertools
import math
import random
import zlib

import torch

from xotorch_support_jetson_amd.inference.shard import Shard
from xotorch_support_jetson_amd.models import weights as W
from xotorch_support_jetson_amd.models.config import from_hf_config, preset
from xotorch_support_jetson_amd.runtime.runner import ShardRunner
from xotorch_support_jetson_amd.train.trainer import ShardTrainer

DEV = "cuda:0"
F64 = torch.float64
MIXED = ("tarepel", "zepalorn")


# ---------------------------------------------------------------------------------------------------------- cases
def listed():
  def decode(name, model, layers, batch, lo, hi):
    return {"name": name, "path": "decode", "model": model, "layers": layers, "batch": batch, "lo": lo, "hi": hi}

  def prompts(name, model, layers, batch, lo, hi, cached=0):
    return {"name": name, "path": "prompts", "model": model, "layers": layers, "batch": batch, "lo": lo, "hi": hi, "cached": cached}

  def generate(name, model, batch, lo, hi, steps):
    return {"name": name, "path": "generate", "model": model, "layers": 4, "batch": batch, "lo": lo, "hi": hi, "steps": steps}
  return [
    # one chat with a small model: every launch and every gap is a user's waiting time
    decode("decode-1b-1", "llama-3.2-1b", 16, 1, 130, 130),
    # a peer of a 4-GPU ring under everyday load: a few dozen conversations of mixed length
    decode("decode-8b-24", "llama-3-8b", 8, 24, 70, 1500),
    # the full batch of the 70B ring (its last peer of 20)
    decode("decode-70b-512", "llama-3-70b", 4, 512, 33, 190),
    # routed experts while a ring decodes: few tokens per expert, expert weights are most of the bytes
    decode("decode-mixtral-64", "mixtral-8x7b", 4, 64, 50, 400),
    # latent attention and many small experts, an odd batch
    decode("decode-deepseek-37", "deepseek-coder-v2-lite", 9, 37, 60, 900),
    # prompts that arrive together, none of a round length
    prompts("prompts-8b-ragged", "llama-3-8b", 8, 9, 17, 1100),
    # one portion of a long document whose beginning is cached
    prompts("prompts-8b-portion", "llama-3-8b", 8, 1, 1999, 1999, cached=8200),
    # one fine-tuning step on a peer of an 8-GPU ring: forward, loss, backward, AdamW
    {"name": "train-8b", "path": "train", "model": "llama-3-8b", "layers": 4, "batch": 2, "length": 1024},
    # mixed-layer designs: a batch of documents read in one step
    prompts("prompts-tarepel", "tarepel", 4, 8, 900, 2600),
    prompts("prompts-zepalorn", "zepalorn", 4, 5, 300, 2100),
    # and whole requests: a short prompt, the answer token by token, the slots returned
    generate("generate-tarepel-48", "tarepel", 48, 9, 90, 24),
    generate("generate-zepalorn-6", "zepalorn", 6, 20, 150, 32),
  ]


def draw(rng):
  def log(lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
  path = rng.choice(("decode", "decode", "decode", "prompts", "prompts", "mixed", "generate", "generate", "train"))
  if path == "decode":
    model, layers = rng.choice((("llama-3.2-1b", 16), ("llama-3-8b", 8), ("llama-3-70b", 4), ("mixtral-8x7b", 4),
                                ("deepseek-coder-v2-lite", 9)))
    batch = log(1, 512)
    lo = log(10, 100)
    return {"path": path, "model": model, "layers": layers, "batch": batch, "lo": lo,
            "hi": max(lo, min(log(60, 4000), 57000 // batch - lo))}
  if path == "prompts":
    model, layers = rng.choice((("llama-3.2-1b", 16), ("llama-3-8b", 8)))
    total, batch, cached = log(40, 3500), rng.randint(1, 12), rng.choice((0, 0, log(20, 9000)))
    hi = max(6, total // batch * 2)
    return {"path": path, "model": model, "layers": layers, "batch": 1 if cached else batch, "lo": max(5, hi // rng.randint(2, 30)),
            "hi": hi, "cached": cached}
  if path == "mixed":
    total, batch = log(60, 13000), rng.randint(1, 12)
    hi = min(2600, max(8, total // batch * 2))
    return {"path": "prompts", "model": rng.choice(MIXED), "layers": 4, "batch": batch, "lo": max(6, hi // rng.randint(2, 20)), "hi": hi,
            "cached": 0}
  if path == "generate":
    batch = log(1, 64)
    lo = log(5, 60)
    return {"path": path, "model": rng.choice(MIXED), "layers": 4, "batch": batch, "lo": lo, "hi": lo + log(10, 120), "steps": rng.randint(12, 32)}
  return {"path": "train", "model": "llama-3-8b", "layers": 4, "batch": rng.randint(1, 3), "length": log(60, 680)}


def _lengths(case):
  """The requests' lengths: spread over [lo, hi] on a log scale, in an order that does not follow the batch."""
  n, lo, hi = case["batch"], case["lo"], case["hi"]
  out = [int(lo * (hi / lo) ** ((i + 0.5) / n)) for i in range(n)]
  random.Random(n).shuffle(out)
  return out


# ---------------------------------------------------------------------------------------------------------- models
def _config(model, layers):
  """ModelConfig, and for the mixed-layer designs the config.json that it was read from."""
  if model not in MIXED:
    return preset(model), None
  D, H, ff = 2048, 16, 5632
  if model == "tarepel":
    par = {"type": "parallel", "mlp": {"kind": "dense", "ff": ff},
           "mixer": {"left": {"heads": H, "kv_heads": 4, "dim": 128, "vdim": 128, "mask": {"size": 1024}, "rot": {"base": 1e6, "dims": 64},
                              "scale": 128 ** -0.5},
                     "right": {"heads": H, "kv_heads": 8, "dim": 128, "vdim": 128, "conv": 4}, "left_scale": 1.0, "right_scale": 1.0}}
    gla = {"type": "gla", "mlp": {"kind": "dense", "ff": ff}, "mixer": {"heads": H, "dim": 64, "vdim": 128, "tau": 16.0, "rank": 16}}
    cfg = {"architecture": "Tarepel", "vocab": 32000, "width": D, "norm": {"eps": 1e-5}, "logit_scale": 1.0,
           "layers": [(par, gla)[i % 2] for i in range(layers)]}
  else:
    mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
    att = {"heads": H, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
           "rot": {"base": 1e6, "dims": 64, "scaling": {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}}}
    kinds = [
      {"type": "channel_delta", "mlp": mlp, "mixer": {"heads": H, "kv_heads": H, "dim": 128, "vdim": 128, "conv": 4, "rank": 128, "gate_rank": 128}},
      {"type": "attention", "mlp": mlp, "mixer": dict(att, mask={"size": 1024, "keep_first": 4})},
      {"type": "parallel", "mlp": mlp,
       "mixer": {"left": dict(att, conv=4, mask={"size": 1024}, softcap=30.0),
                 "right": {"heads": D // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}}}]
    cfg = {"architecture": "Zepalorn", "vocab": 32000, "width": D, "norm": {"eps": 1e-5}, "embedding": {"scale": D ** 0.5},
           "layers": [kinds[(0, 1, 2, 0)[i % 4]] for i in range(layers)]}
  return from_hf_config(cfg), cfg


def _normal(name, shape, std=0.02, mean=0.0):
  """A stored tensor: bf16 values that depend on the name alone."""
  g = torch.Generator(device=DEV).manual_seed(zlib.crc32(name.encode()))
  t = torch.empty(shape, device=DEV, dtype=torch.bfloat16).normal_(0.0, std, generator=g)
  return (t.float() + mean).to(torch.bfloat16) if mean else t


def _decoder_layer(c, model, i):
  """Tensors of decoder layer i by role; expert layers have stacks [E, ...]."""
  D, H, p = c.hidden_size, c.num_heads, f"{model}.{i}."
  out = 0.02 / (2 * c.num_layers) ** 0.5

  def mlp(tag, F, E=0):
    e = (E,) if E else ()
    return {tag + "gate": _normal(p + tag + "gate", e + (F, D)), tag + "up": _normal(p + tag + "up", e + (F, D)),
            tag + "down": _normal(p + tag + "down", e + (D, F), out)}
  t = {"ln1": _normal(p + "ln1", (D,), 0.05, 1.0), "ln2": _normal(p + "ln2", (D,), 0.05, 1.0)}
  if c.is_mla:
    dn, dr, dv, R = c.qk_nope_head_dim, c.qk_rope_head_dim, c.v_head_dim, c.kv_lora_rank
    t.update(qkv=_normal(p + "qkv", (H * (dn + dr) + R + dr, D)), o=_normal(p + "o", (D, H * dv), out), kv_ln=_normal(p + "kv_ln", (R,), 0.05, 1.0),
             uk=_normal(p + "uk", (H, dn, R)), uv=_normal(p + "uv", (H, dv, R)))
  else:
    t.update(qkv=_normal(p + "qkv", ((H + 2 * c.num_kv_heads) * c.head_dim, D)), o=_normal(p + "o", (D, H * c.head_dim), out))
  if c.moe_layer(i):
    t.update(mlp("", c.expert_dim, c.num_experts), router=_normal(p + "router", (c.num_experts, D), 0.1))
    if c.n_shared_experts:
      t.update(mlp("shared.", c.n_shared_experts * c.expert_dim))
  else:
    t.update(mlp("", c.intermediate_size))
  return t


def _decoder_ends(c, model):
  D, V = c.hidden_size, c.vocab_size
  t = {"norm": _normal(model + ".norm", (D,), 0.05, 1.0)}
  t["embed" if c.tie_word_embeddings else "head"] = _normal(model + ".table", (V, D))
  return t


def _mixed_tensors(cfg):
  """Name -> (shape, std, mean) of a mixed-layer checkpoint."""
  D, V, t = cfg["width"], cfg["vocab"], {}

  def proj(name, rows, cols=D):
    t[name] = ((rows, cols), cols ** -0.5, 0.0)

  def norm(name, *shape):
    t[name] = (shape, 0.1, 1.0)
  zep = cfg["architecture"] == "Zepalorn"
  t["embed"] = ((V, D), 0.25 if zep else 1.0, 0.0)
  for i, L in enumerate(cfg["layers"]):
    p, m, kind = f"l{i}.", L["mixer"], L["type"]
    q, left, delta, gla, ssd = p + "mix.", None, None, None, None
    if kind == "parallel":
      left, r = (q + "left.", m["left"]), (q + "right.", m["right"])
      delta, ssd = (None, r) if zep else (r, None)
    elif kind == "attention":
      left = (q, m)
    else:
      delta, gla = ((q, m), None) if zep else (None, (q, m))
    if left:
      n, a = left
      proj(n + "q", a["heads"] * a["dim"]), proj(n + "k", a["kv_heads"] * a["dim"]), proj(n + "o", D, a["heads"] * a["vdim"])
      if zep:
        proj(n + "v", a["kv_heads"] * a["vdim"])
      else:
        t[n + "pb"] = ((a["heads"],), 1.0, -2.0)
      if a.get("conv"):
        for s in "qkv":
          t[n + s + ".conv"] = ((t[n + s][0][0], a["conv"]), 0.5, 0.0)
        norm(n + "q.norm", a["dim"]), norm(n + "k.norm", a["dim"])
    if delta:
      n, r = delta
      for s, rows in (("q", r["kv_heads"] * r["dim"]), ("k", r["kv_heads"] * r["dim"]), ("v", r["heads"] * r["vdim"])):
        proj(n + s, rows)
        t[n + s + ".conv"] = ((rows, r["conv"]), 0.5, 0.0)
      proj(n + "b", r["heads"]), proj(n + "o", D, r["heads"] * r["vdim"]), norm(n + "norm", r["vdim"])
      t[n + "A_log"] = ((r["heads"],), 0.4, -1.2)
      if zep:
        proj(n + "a1", r["rank"]), proj(n + "a2", r["heads"] * r["dim"], r["rank"])
        proj(n + "g1", r["gate_rank"]), proj(n + "g2", r["heads"] * r["vdim"], r["gate_rank"])
        t[n + "dt_bias"] = ((r["heads"] * r["dim"],), 1.0, 0.0)
      else:
        proj(n + "a", r["heads"]), proj(n + "g", r["heads"] * r["vdim"])
        t[n + "dt_bias"] = ((r["heads"],), 1.0, 0.0)
    if gla:
      n, r = gla
      for s, rows in (("q", r["heads"] * r["dim"]), ("k", r["heads"] * r["dim"]), ("v", r["heads"] * r["vdim"]), ("g", r["heads"] * r["vdim"]), ("a1", r["rank"])):
        proj(n + s, rows)
      proj(n + "a2", r["heads"] * r["dim"], r["rank"]), proj(n + "o", D, r["heads"] * r["vdim"]), norm(n + "norm", r["vdim"])
      t[n + "a2.b"] = ((r["heads"] * r["dim"],), 1.0, 3.0)
    if ssd:
      n, s = ssd
      inner, C = s["heads"] * s["vdim"], s["heads"] * s["vdim"] + 2 * s["groups"] * s["state"]
      proj(n + "in", inner + C + s["heads"]), proj(n + "o", D, inner), norm(n + "norm", inner)
      t[n + "conv"], t[n + "conv.b"] = ((C, s["conv"]), 0.5, 0.0), ((C,), 0.5, 0.0)
      t[n + "dt_bias"], t[n + "A_log"], t[n + "D"] = ((s["heads"],), 1.0, 0.0), ((s["heads"],), 0.4, -1.2), ((s["heads"],), 1.0, 0.0)
      norm(q + "left.out", D), norm(q + "right.out", D)
    for n in ("norm1", "norm1b", "norm2", "norm2b") if zep else ("norm1",):
      norm(p + n, *((D,) if zep else ()))
    if not zep:
      t[p + "ls1"], t[p + "ls2"] = ((D,), 0.1, 0.5), ((D,), 0.1, 0.5)
    ff = L["mlp"]["ff"]
    proj(p + "mlp.gate", ff), proj(p + "mlp.up", ff), proj(p + "mlp.down", D, ff)
  norm("final.norm", *((D,) if zep else ()))
  if not zep:
    proj("head", V)
  return t


def _shard(c, model, layers):
  return Shard(model, c.num_layers - layers, c.num_layers - 1, c.num_layers)


def _shard_weights(case):
  model = case["model"]
  c, cfg = _config(model, case["layers"])
  shard = _shard(c, model, case["layers"])
  if cfg is not None:
    spec = _mixed_tensors(cfg)
    return W.mixed_weights(c, shard, lambda n: _normal(f"{model}.{n}", *spec[n]).float().cpu(), DEV, torch.bfloat16)
  sw = W.ShardWeights(c, shard)

  def gated(t, tag=""):
    g, u = t[tag + "gate"], t[tag + "up"]
    return torch.stack([W.interleave_gate_up(a, b) for a, b in zip(g, u)]) if g.dim() == 3 else W.interleave_gate_up(g, u)
  for i in shard.layers():
    t = _decoder_layer(c, model, i)
    lw = sw.layers[i] = W.LayerWeights(t["qkv"], t["o"], gated(t), t["down"], t["ln1"], t["ln2"], router=t.get("router"))
    if c.is_mla:
      lw.kv_ln, lw.wuk, lw.wuv = t["kv_ln"], t["uk"], t["uv"]
    if "shared.gate" in t:
      lw.sh_gu_w, lw.sh_down_w = gated(t, "shared."), t["shared.down"]
  ends = _decoder_ends(c, model)
  sw.norm = ends["norm"]
  sw.lm_head = ends["embed"] if c.tie_word_embeddings else ends["head"]
  if c.tie_word_embeddings:
    sw.embed = ends["embed"]
  return sw


# ---------------------------------------------------------------------------------------------------------- passes
_serving = {}  # the runner in use: a serving process loads its weights, captures its graphs and picks its kernels once
_names = itertools.count()


class _Requests:
  """Requests live on a runner; their pages go back when the caller is done with them."""

  def __init__(self, runner, n):
    self.runner, self.rids = runner, [f"r{next(_names)}" for _ in range(n)]

  def free(self):
    for r in self.rids:
      self.runner.free(r)

  __del__ = free


def _runner(case):
  key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
  if key not in _serving:
    _serving.clear()
    new = case["hi"] + case.get("cached", 0) + case.get("steps", 1) + 1
    pages = sum(-(-(n + case.get("cached", 0) + case.get("steps", 1)) // 64) for n in _lengths(case))
    c, _ = _config(case["model"], case["layers"])
    _serving[key] = [ShardRunner(c, _shard(c, case["model"], case["layers"]), DEV, weights=_shard_weights(case), num_pages=4 * pages + 16,
                                 max_batch=case["batch"], max_ctx=max(2048, -(-new // 64) * 64)), False]
  return _serving[key]


def _inputs(case, seed, n):
  """Inputs of n tokens: ids where the shard holds the embedding, hidden states where it does not."""
  c, _ = _config(case["model"], case["layers"])
  g = torch.Generator(device=DEV).manual_seed(seed)
  if case["layers"] == c.num_layers:
    return torch.randint(0, c.vocab_size, (n,), generator=g, device=DEV, dtype=torch.int32)
  return torch.empty(n, c.hidden_size, device=DEV, dtype=torch.bfloat16).normal_(0.0, 1.0, generator=g)


def prepare(case, seed):
  if case["path"] == "train":
    c, _ = _config(case["model"], case["layers"])
    B, L = case["batch"], case["length"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.empty(B, L, c.hidden_size, device=DEV, dtype=torch.bfloat16).normal_(0.0, 1.0, generator=g)
    y = torch.randint(0, c.vocab_size, (B, L), generator=g, device=DEV)
    return {"trainer": ShardTrainer(_shard_weights(case), DEV, lr=1e-5, max_seq=max(L, 2048)), "x": x, "y": y,
            "lengths": torch.tensor([L - 7 * b for b in range(B)])}
  kept = _runner(case)
  runner, lens = kept[0], _lengths(case)
  req = _Requests(runner, len(lens))
  s = {"runner": runner, "requests": req, "path": case["path"], "cached": case.get("cached", 0), "lens": lens}
  if case["path"] == "decode":
    x = _inputs(case, seed, sum(lens) + len(lens))
    at = 0
    while at < len(lens):  # the conversations so far, some thousand tokens a step
      to, rows = at, 0
      while to < len(lens) and (to == at or rows + lens[to] <= 8192):
        rows += lens[to]
        to += 1
      first = sum(lens[:at])
      runner.forward(req.rids[at:to], lens[at:to], x[first:first + rows])
      at = to
    s["x"] = x[sum(lens):].clone()
  elif case["path"] == "prompts":
    x = _inputs(case, seed, sum(lens) + s["cached"])
    for a in range(0, s["cached"], 4096):
      runner.forward(req.rids, [min(4096, s["cached"] - a)], x[a:min(a + 4096, s["cached"])])
    s["x"] = x[s["cached"]:].clone()
  else:
    x = _inputs(case, seed, sum(lens) + len(lens) * case["steps"])
    s["x"], s["next"] = x[:sum(lens)].clone(), list(x[sum(lens):].view(case["steps"], len(lens)).clone())
  if not kept[1]:  # the server's warm-up
    run(s)
    kept[1] = True
  return s


def run(s):
  if "trainer" in s:
    t = s["trainer"]
    loss, grad_in = t.step("step", s["x"], s["y"], s["lengths"])
    return {"loss": loss, "input": grad_in, **t.grads()}
  runner, rids = s["runner"], s["requests"].rids
  if s["path"] == "decode":
    logits = runner.forward(rids, [1] * len(rids), s["x"])
    for r, n in zip(rids, s["lens"]):
      runner.truncate(r, n)
    return logits
  first = runner.forward(rids, s["lens"], s["x"])
  if s["path"] == "prompts":
    if s["cached"]:
      runner.truncate(rids[0], s["cached"])
    else:
      s["requests"].free()
    return first
  for ids in s["next"]:
    last = runner.forward(rids, [1] * len(rids), ids)
  s["requests"].free()
  return [first, last]


# ---------------------------------------------------------------------------------------------------------- bounds
def work(case):
  c, cfg = _config(case["model"], case["layers"])
  D, V, L = c.hidden_size, c.vocab_size, case["layers"]
  if case["path"] == "train":
    T = case["batch"] * case["length"]
    per = sum(math.prod(s) for s in ((c.qkv_size, D), (D, c.num_heads * c.head_dim), (3 * c.intermediate_size, D)))
    n = L * per + V * D
    # weights twice, gradients and the optimizer's three fp32 values read and written; 3 products per weight
    return {"bytes": n * (2 * 2 + 4 + 6 * 4 + 2) + 4 * T * D, "flops": 6 * T * n + 12 * L * c.num_heads * c.head_dim * T * case["length"] / 2}
  lens, B, cached, steps = _lengths(case), case["batch"], case.get("cached", 0), case.get("steps", 0)
  decode = case["path"] == "decode"
  T = B if decode else sum(lens)
  if cfg is not None:
    spec = _mixed_tensors(cfg)
    n = sum(math.prod(s[0]) for k, s in spec.items() if len(s[0]) == 2 and k not in ("embed", "head"))
    state = pairs = kv = rec = 0
    for lay in cfg["layers"]:
      m = lay["mixer"]
      for a in (m.get("left"), m if lay["type"] == "attention" else None):
        if a:
          size = a["mask"]["size"]
          pairs += a["heads"] * 2 * a["dim"] * sum(k * (k + 1) / 2 if k <= size else size * (k - size / 2) for k in lens)
          kv += a["kv_heads"] * (a["dim"] + a["vdim"]) * 2
      r = m.get("right", m if lay["type"] != "attention" else None)
      if r:
        state += r["heads"] * r.get("dim", r.get("state")) * r["vdim"] * 4
    rec = state / 4 * 6  # decay, read and write of the state, two operations each
    one = 2 * (n + V * D) + B * (2 * state + kv * sum(lens) / B + 4 * V + 4 * D)
    return {"bytes": 2 * (n + V * D) + 4 * T * D + T * kv + B * (state + 4 * V) + steps * one,
            "flops": T * (2 * n + rec) + 2 * pairs + 2 * B * V * D + steps * B * (2 * (n + V * D) + rec)}
  attn = sum(k + 1 for k in lens) if decode else sum(k * (k + 1) / 2 + k * cached for k in lens)
  seen = sum(k + 1 for k in lens) if decode else sum(k + cached for k in lens)
  flops, bytes_ = 2 * B * V * D, 2 * V * D + 4 * B * V
  for i in _shard(c, case["model"], L).layers():
    if c.is_mla:
      H, R, dr, dn, dv = c.num_heads, c.kv_lora_rank, c.qk_rope_head_dim, c.qk_nope_head_dim, c.v_head_dim
      fixed, kv, pair = (H * (dn + dr) + R + dr) * D + D * H * dv + H * (dn + dv) * R, R + dr, 2 * H * (2 * R + dr)
    else:
      fixed, kv, pair = c.qkv_size * D + D * c.num_heads * c.head_dim, 2 * c.num_kv_heads * c.head_dim, 4 * c.num_heads * c.head_dim
    if c.moe_layer(i):
      E, k, F = c.num_experts, c.num_experts_per_tok, c.expert_dim
      fixed += 3 * c.n_shared_experts * F * D + E * D
      hit = E * (1 - (1 - k / E) ** T)  # experts that have a token
      flops += T * 2 * 3 * k * F * D
      bytes_ += 2 * 3 * hit * F * D
    else:
      fixed += 3 * c.intermediate_size * D
    flops += 2 * T * fixed + pair * attn
    bytes_ += 2 * fixed + 2 * kv * (seen + T)
  return {"bytes": bytes_ + 2 * T * D, "flops": flops}


def tolerance(case):
  # Measured against float64, and two orders of the sums differ by no more than twice that: 0.018 after 16 layers on a
  # bf16 residual stream (llama-3.2-1b), 0.007 to 0.009 after the 4 to 9 layers of the other decoders, 0.004 and 0.002 for
  # the designs on an fp32 stream, 0.008 to 0.012 for gradients.  Single values: logits differ like normal noise (five
  # times the mean at most); a token whose experts are almost tied may take another one; gradients span many magnitudes.
  if case["path"] == "train":
    return {"rel": 0.025, "max": 0.5}
  if case["model"] in MIXED:
    return {"rel": 0.012, "max": 0.1}
  if case["model"] == "llama-3.2-1b":
    return {"rel": 0.03, "max": 0.25}
  return {"rel": 0.02, "max": 0.15} if "llama" in case["model"] else {"rel": 0.03, "max": 0.5}


# ---------------------------------------------------------------------------------------------------------- float64
def _rms(x, eps):
  return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _frequencies(dims, base, s):
  """(angles per position [dims / 2], factor on cos and sin): plain, banded (llama3) or YaRN scaling."""
  f = base ** (-torch.arange(0, dims, 2, dtype=F64, device=DEV) / dims)
  if not s:
    return f, 1.0
  if s.get("rope_type") == "llama3":
    turns = s["original_max_position_embeddings"] * f / (2 * math.pi)
    keep = ((turns - s["low_freq_factor"]) / (s["high_freq_factor"] - s["low_freq_factor"])).clamp(0, 1)
    return f * keep + f / s["factor"] * (1 - keep), 1.0
  original = s.get("original", s.get("original_max_position_embeddings"))

  def at(turns):
    return dims * math.log(original / (2 * math.pi * turns)) / (2 * math.log(base))
  lo, hi = max(math.floor(at(s.get("fast", s.get("beta_fast")))), 0), min(math.ceil(at(s.get("slow", s.get("beta_slow")))), dims - 1)
  ramp = ((torch.arange(dims // 2, dtype=F64, device=DEV) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
  return f / s["factor"] * ramp + f * (1 - ramp), 1.0 if "mscale" in s else 0.1 * math.log(s["factor"]) + 1.0


def _rotate(x, first, dims, base, scaling=None, neighbours=False):
  """x [..., n, heads, d], positions from `first`: pairs (i, i + dims / 2), or (2i, 2i + 1)."""
  f, m = _frequencies(dims, base, scaling)
  ang = torch.arange(first, first + x.shape[-3], dtype=F64, device=DEV)[:, None, None] * f
  c, s, out = m * ang.cos(), m * ang.sin(), x.clone()
  a, b = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
  u, v = x[..., a], x[..., b]
  out[..., a], out[..., b] = u * c - v * s, v * c + u * s
  return out


def _attend(q, k, v, scale, sees, cap=0.0, bias=None):
  """One sequence: q [n, H, d] are its last n tokens, k [m, G, d], v [m, G, dv] all of them.  Softmax, or with a bias per
  head a sigmoid per key."""
  (n, H, d), (m, G) = q.shape, k.shape[:2]
  out = []
  for a in range(0, n, 512):
    b = min(a + 512, n)
    at = torch.arange(m - n + a, m - n + b, device=DEV)[:, None]
    ok = sees(at, torch.arange(m, device=DEV)[None, :])
    s = torch.matmul(q[a:b].reshape(b - a, G, H // G, d).permute(1, 2, 0, 3), k.permute(1, 2, 0)[:, None]) * scale
    if cap:
      s = cap * torch.tanh(s / cap)
    if bias is not None:
      p = torch.where(ok, torch.sigmoid(s + bias.view(G, H // G, 1, 1)), 0.0)
    else:
      p = torch.softmax(s.masked_fill(~ok, -math.inf), -1)
    out.append(torch.matmul(p, v.permute(1, 0, 2)[:, None]).permute(2, 0, 1, 3).reshape(b - a, H, -1))
  return torch.cat(out)


def _causal(i, j):
  return j <= i


def _decoder64(c, model, layers, x, spans, tensors):
  """Hidden states [T, D] through the layers; spans: (first, last + 1) row of every sequence."""
  H, G, eps = c.num_heads, c.num_kv_heads, c.rms_norm_eps
  for i in range(c.num_layers - layers, c.num_layers):
    t = tensors(i)
    h = _rms(x, eps) * t["ln1"]
    a = h @ t["qkv"].T
    heads = []
    for s, e in spans:
      if c.is_mla:
        dn, dr, R = c.qk_nope_head_dim, c.qk_rope_head_dim, c.kv_lora_rank
        sc = c.rope_scaling
        scale = (dn + dr) ** -0.5 * (0.1 * sc["mscale_all_dim"] * math.log(sc["factor"]) + 1.0) ** 2
        qn, qr, lat, kr = a[s:e].split([H * dn, H * dr, R, dr], 1)
        lat = _rms(lat, eps) * t["kv_ln"]
        qr = _rotate(qr.reshape(e - s, H, dr), 0, dr, c.rope_theta, sc)
        kr = _rotate(kr.reshape(e - s, 1, dr), 0, dr, c.rope_theta, sc).expand(-1, H, -1)
        k = torch.cat([torch.einsum("tr,hdr->thd", lat, t["uk"]), kr], -1)
        heads.append(_attend(torch.cat([qn.reshape(e - s, H, dn), qr], -1), k, torch.einsum("tr,hdr->thd", lat, t["uv"]), scale, _causal).flatten(1))
      else:
        d = c.head_dim
        q, k, v = a[s:e].split([H * d, G * d, G * d], 1)
        q, k = (_rotate(z.reshape(e - s, -1, d), 0, d, c.rope_theta, c.rope_scaling) for z in (q, k))
        heads.append(_attend(q, k, v.reshape(e - s, G, d), d ** -0.5, _causal).flatten(1))
    x = x + torch.cat(heads) @ t["o"].T
    h = _rms(x, eps) * t["ln2"]

    def gated(h, g, u, d):
      return (torch.nn.functional.silu(h @ g.T) * (h @ u.T)) @ d.T
    if "router" not in t:
      x = x + torch.cat([gated(r, t["gate"], t["up"], t["down"]) for r in h.split(8192)])
      continue
    score = torch.softmax(h @ t["router"].T, -1)
    top, idx = score.topk(c.num_experts_per_tok, -1)
    if c.norm_topk_prob:
      top = top / top.sum(-1, keepdim=True)
    y = gated(h, t["shared.gate"], t["shared.up"], t["shared.down"]) if "shared.gate" in t else torch.zeros_like(x)
    for e in range(c.num_experts):
      row, slot = (idx == e).nonzero(as_tuple=True)
      if row.numel():
        y.index_add_(0, row, gated(h[row], t["gate"][e].to(F64), t["up"][e].to(F64), t["down"][e].to(F64)) * top[row, slot, None])
    x = x + y
  return x


def _conv(u, w, b=None):
  """u [B, T, C], w [C, taps]: causal, the last tap on the current token."""
  y = sum(torch.nn.functional.pad(u, (0, 0, w.shape[1] - 1 - j, 0))[:, :u.shape[1]] * w[:, j] for j in range(w.shape[1]))
  return y if b is None else y + b


def _recur(q, k, v, g, beta, delta):
  """State S [d, dv] per head: S <- g S; S <- S + k u^T with u = beta (v - S^T k) or beta v; o = S^T q.
  q, k [B, T, H, d], v [B, T, H, dv], g [B, T, H, d | 1], beta [B, T, H, 1]."""
  B, T, H, d = q.shape
  S, out = torch.zeros(B, H, d, v.shape[-1], dtype=F64, device=DEV), torch.empty_like(v)
  for t in range(T):
    S *= g[:, t, :, :, None]
    u = beta[:, t] * (v[:, t] - torch.matmul(k[:, t, :, None], S).squeeze(2)) if delta else beta[:, t] * v[:, t]
    S += k[:, t, :, :, None] * u[:, :, None]
    out[:, t] = torch.matmul(q[:, t, :, None], S).squeeze(2)
  return out


def _per_head(x, heads):
  return x.reshape(*x.shape[:2], heads, -1)


def _tarepel64(cfg, t, x, last):
  eps, silu = cfg["norm"]["eps"], torch.nn.functional.silu
  for i, L in enumerate(cfg["layers"]):
    p, m = f"l{i}.", L["mixer"]
    h = _rms(x, eps) * t(p + "norm1")
    if L["type"] == "parallel":
      n, a = p + "mix.left.", m["left"]
      q, raw = _per_head(h @ t(n + "q").T, a["heads"]), _per_head(h @ t(n + "k").T, a["kv_heads"])
      q, k = (_rotate(z, 0, a["rot"]["dims"], a["rot"]["base"]) for z in (q, raw))
      size = a["mask"]["size"]
      o = torch.stack([_attend(q[b], k[b], raw[b], a["scale"], lambda i, j: (j <= i) & (i // size == j // size), bias=t(n + "pb"))
                       for b in range(len(x))])
      y = m["left_scale"] * (o.flatten(2) @ t(n + "o").T)
      n, r = p + "mix.right.", m["right"]
      H, G = r["heads"], r["kv_heads"]
      q, k, v = (silu(_conv(h @ t(n + s).T, t(n + s + ".conv"))) for s in "qkv")
      q, k = (_per_head(z, G) for z in (q, k))
      q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
      q, k = (z.repeat_interleave(H // G, 2) for z in (q * r["dim"] ** -0.5, k))
      g = torch.exp(-torch.exp(t(n + "A_log")) * torch.nn.functional.softplus(h @ t(n + "a").T + t(n + "dt_bias")))
      o = _recur(q, k, _per_head(v, H), g[..., None], torch.sigmoid(h @ t(n + "b").T)[..., None], True)
      scale = m["right_scale"]
    else:
      n, r = p + "mix.", m
      H = r["heads"]
      g = torch.sigmoid((h @ t(n + "a1").T) @ t(n + "a2").T + t(n + "a2.b")) ** (1.0 / r["tau"])
      q, k, v, g = (_per_head(z, H) for z in (h @ t(n + "q").T * r["dim"] ** -0.5, h @ t(n + "k").T, h @ t(n + "v").T, g))
      o = _recur(q, k, v, g, torch.ones_like(v[..., :1]), False)
      y, scale = 0.0, 1.0
    o = _rms(o, eps) * t(n + "norm") * silu(_per_head(h @ t(n + "g").T, H))
    y = y + scale * (o.flatten(2) @ t(n + "o").T)
    f = torch.nn.functional.gelu(h @ t(p + "mlp.gate").T, approximate="tanh") * (h @ t(p + "mlp.up").T)
    x = x + t(p + "ls1") * y + t(p + "ls2") * (f @ t(p + "mlp.down").T)
  return [(_rms(z, eps) * t("final.norm")) @ t("head").T * cfg["logit_scale"] for z in last(x)]


def _zepalorn64(cfg, t, x, last):
  eps, silu = cfg["norm"]["eps"], torch.nn.functional.silu

  def ln(z, w):
    return torch.nn.functional.layer_norm(z, z.shape[-1:], t(w), None, eps)
  for i, L in enumerate(cfg["layers"]):
    p, m, kind = f"l{i}.", L["mixer"], L["type"]
    n, h = p + "mix.", ln(x, p + "norm1")
    if kind == "channel_delta":
      H, G = m["heads"], m["kv_heads"]
      q, k, v = (silu(_conv(h @ t(n + s).T, t(n + s + ".conv"))) for s in "qkv")
      q, k = (_per_head(z, G) for z in (q, k))
      q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
      q, k = (z.repeat_interleave(H // G, 2) for z in (q * m["dim"] ** -0.5, k))
      z = torch.nn.functional.softplus((h @ t(n + "a1").T) @ t(n + "a2").T + t(n + "dt_bias"))
      g = torch.exp(-torch.exp(t(n + "A_log"))[:, None] * _per_head(z, H))
      o = _recur(q, k, _per_head(v, H), g, torch.sigmoid(h @ t(n + "b").T)[..., None], True)
      o = _rms(o, eps) * t(n + "norm") * torch.sigmoid(_per_head((h @ t(n + "g1").T) @ t(n + "g2").T, H))
      y = o.flatten(2) @ t(n + "o").T
    else:
      a = m if kind == "attention" else m["left"]
      l, par, size = (n, False, a["mask"]["size"]) if kind == "attention" else (n + "left.", True, a["mask"]["size"])
      q, k, v = (_per_head(_conv(h @ t(l + s).T, t(l + s + ".conv")) if par else h @ t(l + s).T, a["heads" if s == "q" else "kv_heads"]) for s in "qkv")
      if par:
        q, k = _rms(q, eps) * t(l + "q.norm"), _rms(k, eps) * t(l + "k.norm")
      q, k = (_rotate(z, 0, a["rot"]["dims"], a["rot"]["base"], a["rot"]["scaling"], neighbours=par) for z in (q, k))
      keep = a["mask"].get("keep_first", 0)
      sees = (lambda i, j: (j <= i) & (i // size == j // size)) if par else (lambda i, j: (j <= i) & ((i - j < size) | (j < keep)))
      o = torch.stack([_attend(q[b], k[b], v[b], a["scale"], sees, a.get("softcap", 0.0)) for b in range(len(x))])
      y = o.flatten(2) @ t(l + "o").T
      if par:
        r, s = n + "right.", m["right"]
        H, N, G = s["heads"], s["state"], s["groups"]
        inner = H * s["vdim"]
        z, xbc, dt = (h @ t(r + "in").T).split([inner, inner + 2 * G * N, H], 2)
        u, B, C = silu(_conv(xbc, t(r + "conv"), t(r + "conv.b"))).split([inner, G * N, G * N], 2)
        u, B, C = _per_head(u, H), _per_head(B, G).repeat_interleave(H // G, 2), _per_head(C, G).repeat_interleave(H // G, 2)
        dt = torch.nn.functional.softplus(dt + t(r + "dt_bias"))
        o = _recur(C, B, u, torch.exp(-torch.exp(t(r + "A_log")) * dt)[..., None], dt[..., None], False) + t(r + "D")[:, None] * u
        o = _rms(_per_head(o.flatten(2) * silu(z), s["norm_groups"]), eps).flatten(2) * t(r + "norm")
        y = 0.5 * (_rms(y, eps) * t(n + "left.out") + _rms(o @ t(r + "o").T, eps) * t(n + "right.out"))
    x = x + ln(y, p + "norm1b")
    h, lim = ln(x, p + "norm2"), L["mlp"]["limit"]
    g, u = (h @ t(p + "mlp.gate").T).clamp(max=lim), (h @ t(p + "mlp.up").T).clamp(-lim, lim)
    x = x + ln((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ t(p + "mlp.down").T, p + "norm2b")
  return [ln(z, "final.norm") @ t("embed").T for z in last(x)]


def exact(case, seed):
  c, cfg = _config(case["model"], case["layers"])
  if case["path"] == "train":
    return _train64(case, c, seed)
  lens, B, cached, steps = _lengths(case), case["batch"], case.get("cached", 0), case.get("steps", 0)
  with torch.no_grad():
    if cfg is not None:
      ids = _inputs(case, seed, sum(lens) + B * steps).long()
      seqs = [torch.cat([a, b]) for a, b in zip(ids[:sum(lens)].split(lens), ids[sum(lens):].view(steps, B).T)]
      rows = torch.nn.utils.rnn.pad_sequence(seqs, batch_first=True)  # (later tokens do not reach earlier ones)
      spec, at = _mixed_tensors(cfg), torch.arange(B, device=DEV)

      def t(n):
        return _normal(f"{case['model']}.{n}", *spec[n]).to(F64)

      def last(x):
        return [x[at, torch.tensor(lens, device=DEV) + k - 1] for k in ((0, steps) if steps else (0,))]
      x = t("embed")[rows] * cfg.get("embedding", {}).get("scale", 1.0)
      out = (_tarepel64 if case["model"] == "tarepel" else _zepalorn64)(cfg, t, x, last)
      return out if steps else out[0]
    ends = {k: v.to(F64) for k, v in _decoder_ends(c, case["model"]).items()}
    decode = case["path"] == "decode"
    raw = _inputs(case, seed, sum(lens) + (B if decode else cached))
    if decode:  # every conversation and its new token
      raw = torch.cat([z for a, b in zip(raw[:sum(lens)].split(lens), raw[sum(lens):].split(1)) for z in (a, b)])
    x = ends["embed"][raw.long()] if raw.dim() == 1 else raw.to(F64)
    sizes = [n + (1 if decode else cached) for n in lens]
    stops = list(itertools.accumulate(sizes))

    def tensors(i):
      return {k: v if v.dim() == 3 and k in ("gate", "up", "down") else v.to(F64) for k, v in _decoder_layer(c, case["model"], i).items()}
    x = _decoder64(c, case["model"], case["layers"], x, [(e - n, e) for e, n in zip(stops, sizes)], tensors)
    x = x[torch.tensor(stops, device=DEV) - 1]
    return (_rms(x, c.rms_norm_eps) * ends["norm"]) @ ends["embed" if c.tie_word_embeddings else "head"].T


def _train64(case, c, seed):
  B, L, model = case["batch"], case["length"], case["model"]
  g = torch.Generator(device=DEV).manual_seed(seed)
  x = torch.empty(B, L, c.hidden_size, device=DEV, dtype=torch.bfloat16).normal_(0.0, 1.0, generator=g)
  y = torch.randint(0, c.vocab_size, (B, L), generator=g, device=DEV)
  x = x.to(F64).requires_grad_()
  kept = {i: {k: v.to(F64).requires_grad_() for k, v in _decoder_layer(c, model, i).items()} for i in range(c.num_layers - case["layers"], c.num_layers)}
  ends = {k: v.to(F64).requires_grad_() for k, v in _decoder_ends(c, model).items()}
  h = _decoder64(c, model, case["layers"], x.view(B * L, -1), [(b * L, (b + 1) * L) for b in range(B)], kept.__getitem__)
  valid = torch.cat([torch.arange(b * L, (b + 1) * L - 7 * b, device=DEV) for b in range(B)])
  logits = (_rms(h[valid], c.rms_norm_eps) * ends["norm"]) @ ends["head"].T
  loss = torch.nn.functional.cross_entropy(logits, y.view(-1)[valid])
  loss.backward()
  out = {"loss": float(loss), "input": x.grad, "norm": ends["norm"].grad, "lm_head": ends["head"].grad}
  for i, t in kept.items():
    out.update({f"{i}.{k}": t[k].grad for k in ("qkv", "o", "down", "ln1", "ln2")}, **{f"{i}.gu": torch.cat([t["gate"].grad, t["up"].grad])})
  return out
