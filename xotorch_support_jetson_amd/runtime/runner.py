"""ShardRunner: one pipeline shard on one device — weights, paged KV pool, request bookkeeping,
step-input construction and HIP-graph replay of decode steps.

Requests are independent: each owns pages in the shard's KV pool (native C++ BlockManager), so any
number of sequences can be in flight on a shard and a ring stage can interleave micro-batches.
Decode steps of a given padded batch size are captured once into a HIP graph (torch.cuda.CUDAGraph
is hipGraph on ROCm) and replayed: one host launch per shard step instead of ~10 kernels per layer.
"""
from __future__ import annotations

import os
from typing import Dict, List, Optional, Sequence

import torch

from ..inference.shard import Shard
from ..models.config import ModelConfig
from ..models.transformer import KVCache, ShardModel, StatePool, StepInputs
from ..models.weights import ShardWeights, prepare_for_decode, random_weights
from ..ops import linear as linear_mod

PAGE = 64


def _block_manager(num_pages: int):
  try:
    from .. import _runtime
    return _runtime.BlockManager(num_pages, PAGE)
  except ImportError:
    from .block_manager_py import BlockManager  # pure-python fallback for hosts without the build
    return BlockManager(num_pages, PAGE)


def _slot_manager(slots: int):
  try:
    from .. import _runtime
    return _runtime.SlotManager(slots)
  except (ImportError, AttributeError):
    return SlotManager(slots)  # pure-python twin for hosts without the build


class SlotManager:
  """State slots of models with recurrent layers: one slot per live request, handed out on admission and returned
  when the request ends (lowest free slot first, so a small pool is reused at once).  Python twin of the native
  class (csrc/runtime/slot_manager.h), used where the C++ runtime is not built and as its executable specification."""

  def __init__(self, slots: int):
    self.slots = slots
    self._free: List[int] = list(range(slots - 1, -1, -1))
    self._of: Dict[str, int] = {}

  @property
  def num_free(self) -> int:
    return len(self._free)

  def has(self, rid: str) -> bool:
    return rid in self._of

  def slot(self, rid: str) -> int:
    return self._of[rid]

  def acquire(self, rid: str) -> int:
    if rid in self._of:
      raise ValueError(f"request {rid} already holds a state slot")
    if not self._free:
      raise RuntimeError(f"state slots exhausted: all {self.slots} are held by live requests")
    s = self._of[rid] = self._free.pop()
    return s

  def release(self, rid: str) -> None:
    s = self._of.pop(rid, None)
    if s is not None:
      self._free.append(s)
      self._free.sort(reverse=True)


def _bucket(n: int) -> int:
  for b in (1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 160, 192, 256, 320, 384, 448, 512):
    if n <= b:
      return b
  return n


def _pack_layout(Bp: int, w: int):
  """Byte offsets of a decode step's inputs in one buffer: ({name: (offset, dtype, shape)}, bytes)."""
  out, at = {}, 0
  for name, dt, shape in (("slots", torch.int64, (Bp,)), ("pos", torch.int32, (Bp,)), ("ctx", torch.int32, (Bp,)),
                          ("sslots", torch.int32, (Bp,)), ("tables", torch.int32, (Bp, w))):
    out[name] = (at, dt, shape)
    n = 8 if dt == torch.int64 else 4
    for s in shape:
      n *= s
    at = -(-(at + n) // 16) * 16
  return out, at


def _unpack(buf: torch.Tensor, Bp: int, w: int) -> Dict[str, torch.Tensor]:
  out = {}
  for name, (at, dt, shape) in _pack_layout(Bp, w)[0].items():
    n = 8 if dt == torch.int64 else 4
    for s in shape:
      n *= s
    out[name] = buf[at:at + n].view(dt).view(shape)
  return out


class ShardRunner:
  def __init__(self, config: ModelConfig, shard: Shard, device: torch.device | str = "cpu",
               weights: Optional[ShardWeights] = None, num_pages: Optional[int] = None, max_batch: int = 128,
               max_ctx: int = 4096, kv_mem_fraction: float = 0.85, seed: int = 0, use_graphs: Optional[bool] = None,
               dtype: torch.dtype = torch.bfloat16):
    """dtype: the compute dtype of mixed-layer models (bfloat16, or float32 for an all-fp32 run: fp32 weights, caches
    and vendor SGEMMs); the other architectures serve in bfloat16 only."""
    self.config = config
    self.dtype = dtype
    if dtype != torch.bfloat16 and not config.is_mixed:
      raise ValueError(f"{config.model_type} serves in bfloat16 only")
    self.shard = shard
    self.device = torch.device(device)
    if self.device.type == "cuda":
      torch.cuda.set_device(self.device)
    self._random_weights, self._seed = weights is None, seed
    self.weights = weights if weights is not None else random_weights(config, shard, self.device, seed=seed,
                                                                      **({"dtype": dtype} if config.is_mixed else {}))
    if self.device.type == "cuda" and os.environ.get("XOT_SHUFFLE", "1") == "1":
      # projection weights -> pre-shuffled MFMA-fragment layout: gemm_stream for decode-shaped M, gemm_big
      # (256 x 256 LDS-DMA tiles, fused SiLU / residual epilogues) for large decode batches and prefill
      # chunks -- every projection runs on the library's own kernels (XOT_ROWMAJOR_PROJ=gu,... keeps the
      # named projections row-major for A/B runs against the vendor GEMM)
      env = os.environ.get("XOT_ROWMAJOR_PROJ")
      keep = [p for p in env.split(",") if p] if env is not None else []
      # XOT_WEIGHT_DTYPE=fp8: weight-only e4m3 projections (half the bytes per decode step; opt-in, the
      # serving default and every benchmark headline stay bf16)
      self.weight_dtype = os.environ.get("XOT_WEIGHT_DTYPE", "bf16")
      prepare_for_decode(self.weights, keep_rowmajor=keep, fp8=self.weight_dtype == "fp8")
    n_layers = shard.get_layer_count()
    per_page = KVCache.bytes_per_page(config, n_layers, shard.layers(), torch.empty(0, dtype=dtype).element_size()) \
      if config.is_mixed else KVCache.bytes_per_page(config, n_layers)
    if num_pages is None:
      if self.device.type == "cuda":
        free, _ = torch.cuda.mem_get_info(self.device)
        reserve = 4 << 30  # activations, workspaces, graphs
        num_pages = int(max(free - reserve, per_page * 64) * kv_mem_fraction) // per_page
      else:
        num_pages = max(64, (max_batch * max_ctx) // PAGE // 4)
      num_pages = min(num_pages, max_batch * (-(-max_ctx // PAGE)) + 16)
    self.kv = KVCache(config, n_layers, num_pages, self.device, dtype, shard.layers()) if config.is_mixed else \
      KVCache(config, n_layers, num_pages, self.device)
    self.bm = _block_manager(num_pages)
    # recurrent layers: one state slot per live request (max_batch of them), cleared on admission
    self.sm = _slot_manager(max_batch) if config.has_state else None
    self.state = StatePool(config, shard.layers(), max_batch, self.device) if config.has_state else None
    self.max_ctx = max_ctx
    self.max_batch = max_batch
    self.width = -(-max_ctx // PAGE)
    self.model = ShardModel(self.weights, self.kv, max_batch=max_batch, max_ctx=max_ctx)
    self.model.state = self.state
    if use_graphs is None:
      # MoE routing runs on the device too (moe_route + grouped GEMMs), so every model is capturable
      use_graphs = self.device.type == "cuda" and os.environ.get("XOT_GRAPHS", "1") == "1"
      if dtype == torch.float32 and config.is_mixed and any(s.ffn is not None and s.ffn.experts for s in config.layer_specs):
        use_graphs = False  # an all-fp32 run groups the experts' rows on the host (vendor SGEMM per expert)
    self.use_graphs = use_graphs
    self._graphs: Dict[tuple, dict] = {}
    # decode graphs per (batch bucket, block-table width class): a step whose longest context fits a narrower
    # table replays a graph captured with it, so the split-KV partitioning (chosen from the table width,
    # static per graph) follows the contexts actually served instead of max_ctx -- at max_ctx 8192 and
    # contexts of a few hundred tokens the full width split every sequence into 4 mostly empty partitions
    # plus a merge pass
    # (16 pages: the widest table the 8-wave single-partition attention takes at small batch, ops/kernels.py)
    self._widths = sorted({w for w in (8, 16, 32) if w < self.width} | {self.width})
    # host staging of the step inputs, double-buffered: a step's async copies read one set while the host
    # fills the other for the next step, so the host can queue a step behind the one still copying (with
    # one set it had to wait for the previous step's copies before writing the next step's inputs)
    bmax = _bucket(max_batch)
    self._sets = []
    for _ in range(2):
      st = {"tables": torch.zeros(max_batch, self.width, dtype=torch.int32),
            "ctx": torch.zeros(max_batch, dtype=torch.int32),
            # a decode step's inputs as its graph holds them, one copy for all (each copy costs the step 3 to 5 us)
            "pack": torch.zeros(_pack_layout(bmax, self.width)[1], dtype=torch.uint8)}
      if self.device.type == "cuda":
        # pinned: an async copy out of pageable memory may wait for the stream to drain, i.e. for the step
        # already running, which would forbid queueing the next decode step behind it
        st = {k: v.pin_memory() for k, v in st.items()}
      st["views"] = {}  # of the pack, per captured (batch bucket, table width)
      st["event"] = None  # completion of the last async H2D copy out of this set
      self._sets.append(st)
    self._set_idx = 1
    self._use_set(0)

  def _use_set(self, i: int) -> None:
    st = self._sets[i]
    self._set_idx = i
    self._tables_host, self._ctx_host, self._pack_host = st["tables"], st["ctx"], st["pack"]

  def _reuse_staging(self) -> None:
    """Switch to the other staging set; wait only if ITS last async copy (two steps back) is still running."""
    i = self._set_idx ^ 1
    ev = self._sets[i]["event"]
    if ev is not None:
      ev.synchronize()
      self._sets[i]["event"] = None
    self._use_set(i)

  def _mark_staged(self) -> None:
    if self.device.type == "cuda":
      ev = torch.cuda.Event()
      ev.record()
      self._sets[self._set_idx]["event"] = ev

  @property
  def hidden_dtype(self) -> torch.dtype:
    """dtype of the hidden states that travel between shards (mixed-layer models carry an fp32 residual stream)."""
    return torch.float32 if self.config.is_mixed else torch.bfloat16

  # ------------------------------------------------------------------ bookkeeping
  def has(self, rid: str) -> bool:
    return self.bm.has(rid)

  def num_tokens(self, rid: str) -> int:
    return self.bm.num_tokens(rid) if self.bm.has(rid) else 0

  def free(self, rid: str) -> None:
    self.bm.free(rid)
    if self.sm is not None:
      self.sm.release(rid)

  def can_admit(self, rid: str, n_new: int) -> bool:
    if self.sm is not None and not self.sm.has(rid) and self.sm.num_free == 0:
      return False
    return self.bm.can_append(rid, n_new) and self.num_tokens(rid) + n_new <= self.max_ctx

  def _state_slots(self, rids: Sequence[str]) -> List[int]:
    """The requests' state slots; requests seen for the first time get cleared ones."""
    out, new = [], []
    try:
      for rid in rids:
        if self.sm.has(rid):
          out.append(self.sm.slot(rid))
          continue
        if self.bm.has(rid) and self.bm.num_tokens(rid) > 0:
          raise RuntimeError(f"request {rid} holds cached tokens but no recurrent state")
        out.append(self.sm.acquire(rid))
        new.append(out[-1])
    finally:  # (also where a later request is refused: those before it keep their slots)
      if new:
        self.state.clear(new)
    return out

  def truncate(self, rid: str, n: int) -> None:
    if self.sm is not None and n != self.num_tokens(rid):
      raise RuntimeError("a recurrent state cannot be rolled back to an earlier token")
    self.bm.truncate(rid, n)

  # ------------------------------------------------------------------ step inputs
  def _prepare(self, rids: Sequence[str], qlens: Sequence[int], logit_rows: Optional[Sequence[int]] = None) -> StepInputs:
    if len(rids) > self.max_batch:
      raise ValueError(f"batch {len(rids)} exceeds max_batch {self.max_batch}")
    self._reuse_staging()
    pos: List[int] = []
    slots: List[int] = []
    cu = [0]
    sslots = self._state_slots(rids) if self.sm is not None else None
    for rid, n in zip(rids, qlens):
      start = self.num_tokens(rid)
      if start + n > self.max_ctx:
        raise ValueError(f"request {rid}: context {start + n} exceeds max_ctx {self.max_ctx}")
      slots += self.bm.append(rid, n)
      pos += self.model.rope_pos(start, n)
      cu.append(cu[-1] + n)
    if logit_rows is not None and any(not 0 <= r < cu[-1] for r in logit_rows):
      raise ValueError("logit_rows must index the step's tokens")
    B = len(rids)
    self.bm.fill_batch(list(rids), self._tables_host[:B].numpy(), self._ctx_host[:B].numpy())
    dev = self.device
    nb = non_blocking = dev.type == "cuda"
    inp = StepInputs(
      positions=torch.tensor(pos, dtype=torch.int32).to(dev, non_blocking=nb),
      slots=torch.tensor(slots, dtype=torch.int64).to(dev, non_blocking=nb),
      block_tables=self._tables_host[:B].to(dev, non_blocking=non_blocking),
      ctx_lens=self._ctx_host[:B].to(dev, non_blocking=non_blocking),
      cu_q=torch.tensor(cu, dtype=torch.int32).to(dev, non_blocking=nb),
      last_idx=torch.tensor([c - 1 for c in cu[1:]] if logit_rows is None else list(logit_rows),
                            dtype=torch.int64).to(dev, non_blocking=nb),
      max_qlen=max(qlens),
      decode=all(q == 1 for q in qlens),
      state_slots=None if sslots is None else torch.tensor(sslots, dtype=torch.int32).to(dev, non_blocking=nb),
      all_rows=logit_rows is None and all(q == 1 for q in qlens),
    )
    self._mark_staged()
    return inp

  # ------------------------------------------------------------------ forward
  def forward(self, rids: Sequence[str], qlens: Sequence[int], x: torch.Tensor,
              image_embeds: Optional[torch.Tensor] = None, logit_rows: Optional[Sequence[int]] = None) -> torch.Tensor:
    """Run this shard for the given requests.  x = token ids [sum(qlens)] (first shard) or hidden
    [sum(qlens), D].  Allocates KV slots for the new tokens.  Returns hidden [T, D] or, on the last
    shard, fp32 logits [len(rids), V] of each request's last token.  image_embeds (LLaVA, first shard):
    projected image features for the image-token rows of x, in order.
    logit_rows (last shard): rows of x whose logits to return instead of each request's last token's, [len(logit_rows), V]
    (replaying recorded traffic, scoring a prompt)."""
    x = x.to(self.device, non_blocking=True)
    if (self.use_graphs and image_embeds is None and logit_rows is None and all(q == 1 for q in qlens)
        and len(rids) <= self.max_batch):
      return self._decode_graph(rids, x)
    inp = self._prepare(rids, qlens, logit_rows)
    if image_embeds is not None:
      inp.image_embeds = image_embeds.to(self.device)
    return self.model.forward(x, inp)

  def image_features(self, pixels: torch.Tensor) -> torch.Tensor:
    """LLaVA first shard: [N, 3, S, S] pixel batch -> [N * image tokens, D] projected features."""
    from ..models.vision import image_features
    if self.weights.vision is None:
      raise ValueError(f"{self.shard.model_id}: this shard has no vision tower")
    with torch.inference_mode():
      return image_features(self.config, self.weights.vision, pixels.to(self.device))

  # ------------------------------------------------------------------ graphs
  def _pack_views(self, Bp: int, w: int) -> dict:
    """numpy views of the current staging set's pack as the graph (Bp, w) lays it out, and its length in bytes."""
    views = self._sets[self._set_idx]["views"]
    v = views.get((Bp, w))
    if v is None:
      v = views[(Bp, w)] = {k: t.numpy() for k, t in _unpack(self._pack_host, Bp, w).items()}
      v["bytes"] = _pack_layout(Bp, w)[1]
    return v

  def _decode_graph(self, rids: Sequence[str], x: torch.Tensor) -> torch.Tensor:
    B = len(rids)
    Bp = min(_bucket(B), self.max_batch)
    # host bookkeeping -> static buffers
    self._reuse_staging()
    pos, slots = [], []
    most = 0
    sslots = self._state_slots(rids) if self.sm is not None else None
    for rid in rids:
      start = self.num_tokens(rid)
      if start + 1 > self.max_ctx:
        raise ValueError(f"request {rid}: context exceeds max_ctx {self.max_ctx}")
      slots += self.bm.append(rid, 1)
      pos += self.model.rope_pos(start, 1)
      most = max(most, start + 1)
    need = -(-most // PAGE)
    w = next(c for c in self._widths if c >= need)
    g = self._graphs.get((Bp, w))
    if g is None:
      g = self._capture(Bp, w)
    v = self._pack_views(Bp, w)
    self.bm.fill_batch(list(rids), v["tables"][:B], v["ctx"][:B])
    v["pos"][:B], v["slots"][:B] = pos, slots
    v["sslots"][:B] = -1 if sslots is None else sslots
    # (padding rows: no context, no KV or state slot)
    v["tables"][B:], v["ctx"][B:], v["pos"][B:], v["slots"][B:], v["sslots"][B:] = 0, 0, 0, -1, -1
    g["pack"].copy_(self._pack_host[:v["bytes"]], non_blocking=True)
    self._mark_staged()
    if self.shard.is_first_layer():
      g["x"][:B].copy_(x.view(-1))
      if Bp > B:
        g["x"][B:].zero_()
    else:
      g["x"][:B].copy_(x)
    g["graph"].replay()
    out = g["out"]
    return tuple(t[:B] for t in out) if isinstance(out, tuple) else out[:B]

  # ------------------------------------------------------------------ split LM head
  def head_tail(self, rows_from: int) -> Optional[torch.Tensor]:
    """LM-head rows [rows_from, V) in the device layout, for a first stage that applies them to the
    normed hidden state the last stage sends (parallel/pipeline.py).  None when they cannot be derived
    here (externally loaded weights without the head on this shard)."""
    from ..models.weights import random_head_rows
    w = self.weights
    c = self.config
    if w.lm_head is not None:
      full = w.lm_head
    elif c.tie_word_embeddings and w.embed is not None:
      full = w.embed
    elif self._random_weights:
      full = None
    else:
      return None
    if full is not None:
      t = full[rows_from:]
      if linear_mod.layout_of(full) == "stream":  # rows [r, V) of the shuffled layout: a storage suffix
        t.xot_layout = "stream"
        return t
      return linear_mod.to_stream_layout(t.contiguous())
    t = random_head_rows(c, rows_from, self.device, seed=self._seed)
    return linear_mod.to_stream_layout(t)

  def _capture(self, Bp: int, w: Optional[int] = None) -> dict:
    dev = self.device
    c = self.config
    w = w or self.width
    pack = torch.zeros(_pack_layout(Bp, w)[1], dtype=torch.uint8, device=dev)
    g = {
      "pack": pack, **_unpack(pack, Bp, w),
      "cu": torch.arange(Bp + 1, dtype=torch.int32, device=dev),
      "last": torch.arange(Bp, dtype=torch.int64, device=dev),
    }
    if self.shard.is_first_layer():
      g["x"] = torch.zeros(Bp, dtype=torch.int32, device=dev)
    else:
      g["x"] = torch.zeros(Bp, c.hidden_width, dtype=self.hidden_dtype, device=dev)
    # warm-up and capture run on padding rows only (state slot -1, no KV slot): no request's state is touched
    g["slots"].fill_(-1)
    g["sslots"].fill_(-1)
    inp = StepInputs(g["pos"], g["slots"], g["tables"], g["ctx"], g["cu"], g["last"], 1, True, all_rows=True)
    if self.sm is not None:
      inp.state_slots = g["sslots"]
    # warm up eagerly (also settles the GEMM policy for these shapes) on a side stream
    s = torch.cuda.Stream(dev)
    s.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(s):
      for _ in range(2):
        self.model.forward(g["x"], inp)
    torch.cuda.current_stream(dev).wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    linear_mod.policy.capturing = True
    try:
      # thread-local capture: the process-group watchdog thread keeps polling its RCCL events while
      # this thread captures (global mode would make those queries fail)
      with torch.cuda.graph(graph, capture_error_mode="thread_local"):
        g["out"] = self.model.forward(g["x"], inp)
    finally:
      linear_mod.policy.capturing = False
    g["graph"] = graph
    self._graphs[(Bp, w)] = g
    return g
