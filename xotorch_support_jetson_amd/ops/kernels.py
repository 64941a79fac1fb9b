"""Python entry points of the gfx950 kernel library.

Each function takes torch tensors, allocates outputs when the caller did not preallocate them, and
dispatches to the HIP kernel for GPU tensors or to the fp32 torch reference (`ops.reference`) for
CPU tensors.  GPU tensors never take the reference path: if the extension is missing the call
raises (see `ops._ext.require`).
"""
from __future__ import annotations

import os

import torch

from . import reference as ref
from ._ext import require

EPI = {"none": 0, "resid": 1, "silu": 2, "clamp_glu": 3, "relu2": 4, "gelu_glu": 5}
GLU_EPI = ("silu", "clamp_glu", "gelu_glu")  # epilogues that turn interleaved (gate, up) columns into half as many
PAGE = 64


def _gpu(t: torch.Tensor) -> bool:
  if t.is_cuda:
    require()
    return True
  return False


# ------------------------------------------------------------------ norms / elementwise
def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float, residual: torch.Tensor | None = None,
            out: torch.Tensor | None = None, residual_out: torch.Tensor | None = None):
  """Returns (out, residual_out).  With `residual`, residual_out = x + residual (the new stream)."""
  if not _gpu(x):
    y, r = ref.rmsnorm(x, w, eps, residual)
    if out is not None:
      out.copy_(y)
      y = out
    if residual_out is not None and r is not None:
      residual_out.copy_(r)
      r = residual_out
    return y, r
  out = torch.empty_like(x) if out is None else out
  if residual is not None and residual_out is None:
    residual_out = torch.empty_like(x)
  require().rmsnorm(x, w, out, residual, residual_out, float(eps))
  return out, residual_out


def embedding(ids: torch.Tensor, table: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
  if not _gpu(table):
    y = table[ids.long().clamp(0, table.shape[0] - 1)]
    if out is not None:
      out.copy_(y.reshape(out.shape))
      return out
    return y
  ids32 = ids.to(torch.int32).contiguous()
  out = torch.empty(ids32.numel(), table.shape[1], dtype=table.dtype, device=table.device) if out is None else out
  require().embedding(ids32, table, out)
  return out


def silu_mul(gu: torch.Tensor, out: torch.Tensor | None = None, interleaved16: bool = False) -> torch.Tensor:
  """silu(gate) * up.  gu = [gate | up] halves, or 16-column interleaved tiles (fused gate_up layout)."""
  if not _gpu(gu):
    if interleaved16:
      M, N = gu.shape
      g = gu.view(M, N // 32, 2, 16)
      y = (torch.nn.functional.silu(g[:, :, 0].float()) * g[:, :, 1].float()).reshape(M, N // 2).to(gu.dtype)
    else:
      y = ref.silu_mul(gu)
    if out is not None:
      out.copy_(y)
      return out
    return y
  Fd = gu.shape[-1] // 2
  out = torch.empty(*gu.shape[:-1], Fd, dtype=gu.dtype, device=gu.device) if out is None else out
  require().silu_mul(gu.contiguous(), out, bool(interleaved16))
  return out


# ------------------------------------------------------------------ GEMM
def gemm(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None, residual: torch.Tensor | None = None,
         epi: str = "none", out: torch.Tensor | None = None, out_dtype: torch.dtype | None = None, algo: int = 0,
         nt: int = 0) -> torch.Tensor:
  """y = x @ w.T (+bias) with fused epilogue: 'none' | 'resid' (y += residual) | 'silu'.

  For 'silu' the weight rows must be gate/up interleaved in 16-row tiles (see
  models.weights.interleave_gate_up); the output has w.shape[0] // 2 columns.
  """
  M, N = x.shape[0], w.shape[0]
  ncol = N // 2 if epi == "silu" else N
  if not _gpu(x):
    y = ref.linear(x, w, bias)
    if epi == "silu":
      y = y.view(M, N // 32, 2, 16)
      y = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(M, ncol)
    elif epi == "resid":
      y = y + residual.float()
    dt = out_dtype or (out.dtype if out is not None else x.dtype)
    if out is not None:
      out.copy_(y.to(out.dtype))
      return out
    return y.to(dt)
  if out is None:
    out = torch.empty(M, ncol, dtype=out_dtype or x.dtype, device=x.device)
  if nt == 0:
    nt = 2 if (N // 32) >= 1024 else 1
  if algo == 0 and epi != "silu" and N % 16:  # the skinny kernel tiles 16 output columns; the tiled one masks
    algo = 2
  require().gemm(x, w, out, bias, residual, EPI[epi], int(algo), int(nt))
  return out


# ------------------------------------------------------------------ RoPE + paged KV
def rope_kv_write(qkv: torch.Tensor, pos: torch.Tensor, cos_sin: torch.Tensor, slots: torch.Tensor,
                  k_cache: torch.Tensor, v_cache: torch.Tensor, H: int, Hkv: int,
                  q_out: torch.Tensor | None = None) -> torch.Tensor:
  """qkv [T, (H+2Hkv)*Dh] -> rotated q [T, H, Dh]; rotated k and v written into the paged caches."""
  T = qkv.shape[0]
  Dh = k_cache.shape[-1]
  if not _gpu(qkv):
    x = qkv.view(T, H + 2 * Hkv, Dh)
    q = ref.rope(x[:, :H], pos, cos_sin)
    k = ref.rope(x[:, H:H + Hkv], pos, cos_sin)
    ref.write_kv(k, x[:, H + Hkv:], slots, k_cache, v_cache)
    if q_out is not None:
      q_out.copy_(q.view(q_out.shape))
      return q_out
    return q
  q_out = torch.empty(T, H, Dh, dtype=qkv.dtype, device=qkv.device) if q_out is None else q_out
  require().rope_kv_write(qkv, pos, cos_sin, slots, q_out, k_cache, v_cache, int(H), int(Hkv))
  return q_out


def rope_apply(x: torch.Tensor, pos: torch.Tensor, cos_sin: torch.Tensor, nh: int, Dh: int, inverse: bool = False,
               out: torch.Tensor | None = None) -> torch.Tensor:
  """x [T, >= nh*Dh] (2-D rows) -> rotated copy (or into `out`)."""
  if not _gpu(x):
    y = ref.rope(x[:, :nh * Dh].reshape(-1, nh, Dh), pos, cos_sin, inverse).reshape(x.shape[0], nh * Dh)
    if out is not None:
      out[:, :nh * Dh].copy_(y)
      return out
    return y
  out = torch.empty(x.shape[0], nh * Dh, dtype=x.dtype, device=x.device) if out is None else out
  require().rope_apply(x, out, pos, cos_sin, int(nh), int(Dh), bool(inverse))
  return out


# ------------------------------------------------------------------ attention
# 0: workgroup per (sequence, KV head, partition), waves split pages + LDS combine (scores by rows, P through LDS)
# 1: wave per (sequence, KV head, partition), transposed S^T (lane = query head), no LDS; 5 / 6: the same with the next page's
#    loads under the current one (6: non-temporal)
# 2 / 3: four waves per (sequence, KV head, partition), each as in 5, meeting in LDS (one over short tables at large batches); 3
#    with non-temporal K / V loads
# -1 (default): 0 below 16 (sequence, KV head) pairs; else 3 once a layer's K / V pages (batch x block-table width) outgrow the
#    256 MB last-level cache (256 sequences of 1900 tokens: 301 us, 331 with plain loads), 2 below (24 up to 1407 tokens: 21.3
#    us, 23.5 with nt).  From 16 pairs on 2 also leads 0: 2 sequences x 8 heads of 130 tokens 6.3 us / 9.1, of 8000 21.0 / 29.8;
#    6 of 2000 15.0 / 18.8.  Beside it, without routed experts: a lone sequence is always cut by its length (LONE), and from 16
#    pairs on ragged contexts by theirs (plan_pays), in units of four waves as in 2 / 3
# 7 / 8: as 5 / 6 with two register sets, one wave a SIMD.  With routed experts (DecodeWorkspace.routed) -1 is 0 below 64 pairs
#    and 7 or 8 above: those sum a partition page by page and merge the partitions in order.  2 / 3 deal a context's pages to
#    waves, sums in another order, no less exact; but a token whose experts are almost tied turns on the last bits, and its whole
#    row with it.  So routed models keep the order they have always been served with (64 sequences x 8 heads up to 393 tokens:
#    18.7 us in 8 with its merge, 15.8 in 2)
DECODE_ALGO = int(os.environ.get("XOT_ATTN_DECODE", "-1"))


NT_MIN_KV_BYTES = 256 << 20  # K / V bytes per layer from which the page loads go non-temporal (algo 3)


def resolve_decode_algo(batch: int, Hkv: int, algo: int | None = None, kv_bytes: int | None = None,
                        routed: bool = False) -> int:
  algo = DECODE_ALGO if algo is None else algo
  if algo < 0:
    if batch * Hkv < (64 if routed else 16):
      return 0
    return (7 if routed else 2) + int(kv_bytes is None or kv_bytes >= NT_MIN_KV_BYTES)
  return algo


def group_parts(batch: int, Hkv: int, pages: int) -> int:
  """Most partitions of a context of `pages` pages for algo 2 / 3 (grows with pages)."""
  pairs = max(batch * Hkv, 1)
  if pages <= 8:
    return 1
  return min(max(256 // pairs, 2 if pages > 64 and pairs < 384 else 1), -(-pages // 4))


def choose_pages_per_part(batch: int, Hkv: int, max_ctx: int, algo: int | None = None) -> int:
  """KV pages per split-KV partition for a decode step of `batch` sequences."""
  algo = resolve_decode_algo(batch, Hkv, algo)
  pages = max(1, -(-max_ctx // PAGE))
  if algo == 0:  # enough workgroups to cover 256 CUs several times, >= 4 pages (one per wave) each
    for ppp in (16, 8, 4):
      if batch * Hkv * -(-pages // ppp) >= 1024:
        return ppp
    return 4
  if algo in (2, 3):
    # four waves per unit (csrc/attention.hip attn_decode_group_kernel): a context of 8 pages is two pages a wave and best left
    # whole; longer ones are cut while the units stay within one a CU, in partitions of at least 4 pages (8 sequences x 8 heads, up
    # to 1900 tokens: 20.4 us whole, 13.9 in 4; 16: 21.7, 18.0 in 2, 19.5 in 4; 24: 21.3 whole, 23.0 in 2; more units than CUs
    # share some CUs, and those end the launch: 12 of 900 tokens 19.1 in 3, 15.2 in 2; 20 of 523 20.6 in 2, 13.7 whole), and very
    # long ones once more, since the longest workgroup ends the launch (32 sequences up to 7800 tokens: 100 us whole, 87 in 2)
    return -(-pages // group_parts(batch, Hkv, pages))
  # one wave per unit: ~1024 waves (4 per CU), partitions of 2..32 pages (tools/bench_attn_small.py,
  # profiles/bench_attn_small_r1.json: 2048 waves of shorter partitions lose to the extra merge work)
  nparts = max(1, min(max(pages // 2, 1), -(-1024 // max(batch * Hkv, 1))))
  nparts = max(nparts, -(-pages // 32))
  return -(-pages // nparts)


LONE = object()  # the plan of one sequence
SPLIT_MIN_PAGES = 8  # widest block table whose contexts are not worth cutting


def plan_pays(batch: int, Hkv: int, width_pages: int) -> bool:
  """Whether a decode step cuts its contexts by their lengths (one small launch of 4.5 us a step, then every layer gains).  Up to 8 pages
  a context is two rounds of a unit's four waves and best left whole (20 sequences x 8 heads up to 469 tokens 9.9 us either way).  Beyond,
  the longest context ends the launch unless the pairs fill the chip several times over.  us a layer, uncut (or cut by the table's
  width) / by the lengths: 24 sequences x 8 heads of 128, 74 .. 1407 tokens 21.1 / 15.2 (table of 128 pages 26.4 / 15.8), 8 of 125 .. 3176
  33.5 / 12.8, 32 of 315 .. 7412 114 / 62, 48 of 31 .. 1059 24.4 / 19.8, 128 of 30 .. 1869 68 / 53; even ones 24 of 520 14.0 / 14.1, 64 of
  1000 47.1 / 47.0, 12 of 900 15.3 / 15.0.  More pairs: 256 of 30 .. 1884 107 / 107, 130 of 10 .. 590 26.7 / 26.1."""
  pairs = batch * Hkv
  return width_pages > SPLIT_MIN_PAGES and pairs < 64 * min(width_pages, 32) and pairs * width_pages < 1 << 30


def split_places(batch: int, Hkv: int, width_pages: int) -> int:
  """Places of a plan (csrc/kernels.h decode_split_places), each with a row of partials per query head."""
  return min(batch + 512 // Hkv, batch * -(-width_pages // 4))


class DecodeWorkspace:
  """Split-KV scratch for attn_decode, sized for every batch up to max_batch at this context bound.
  The partitioning is chosen per call from the actual batch (static per captured graph).  routed: the model has routed
  experts (see DECODE_ALGO)."""

  def __init__(self, max_batch: int, H: int, Dh: int, max_ctx: int, device, pages_per_part: int | None = None,
               algo: int | None = None, routed: bool = False):
    self.algo = DECODE_ALGO if algo is None else algo
    self.routed = routed
    self.max_ctx = max_ctx
    self.Hkv_hint = None
    self.Dh = Dh
    self.fixed_ppp = pages_per_part
    pages = max(1, -(-max_ctx // PAGE))
    worst = 1
    for b in range(1, max_batch + 1):
      for hkv in (1, 2, 4, 8, 16):
        kind = resolve_decode_algo(b, hkv, self.algo, routed=routed)
        if pages_per_part is None and kind in (2, 3):
          worst = max(worst, b * group_parts(b, hkv, pages))  # (narrower tables have no more partitions)
          continue
        ppp = pages_per_part or choose_pages_per_part(b, hkv, max_ctx, kind)
        worst = max(worst, b * -(-pages // ppp))
    # rows of split-KV partials: batch * nparts, or the places of a plan (a KV head has at most 16 query heads)
    self.max_batch = max_batch
    self.units = worst  # max over batch of batch * nparts
    if not routed:
      worst = max(worst, split_places(max_batch, max(1, -(-H // 16)), pages))
    self.places = worst
    self.tickets = torch.zeros(max_batch * H, dtype=torch.int32, device=device)
    self.o = torch.empty(worst * H * Dh, dtype=torch.float32, device=device)
    self.ml = torch.empty(worst * H * 2, dtype=torch.float32, device=device)

  def partition(self, batch: int, Hkv: int, width_pages: int):
    """(pages per partition, partitions, kernel) for this call."""
    algo = resolve_decode_algo(batch, Hkv, self.algo, batch * Hkv * width_pages * PAGE * self.Dh * 4, self.routed)
    ppp = self.fixed_ppp or choose_pages_per_part(batch, Hkv, width_pages * PAGE, algo)
    nparts = max(1, -(-width_pages // ppp))
    if batch * nparts > self.units:
      raise RuntimeError(f"decode workspace sized for {self.units} units, need {batch * nparts}")
    return ppp, nparts, algo


  def plan(self, block_tables: torch.Tensor, ctx_lens: torch.Tensor, Hkv: int):
    """The units of a decode step's attention (csrc/attention.hip decode_plan_kernel), one launch for all layers of the step; LONE for
    one sequence, which needs none; None where attn_decode goes by itself."""
    B, width = ctx_lens.shape[0], block_tables.shape[1]
    if not block_tables.is_cuda or self.fixed_ppp or self.routed or B > self.max_batch or self.Dh not in (64, 128):
      return None
    if split_places(B, Hkv, width) > self.places:  # (tables wider than this workspace's context bound)
      return None
    if B == 1 and self.algo == -1 and width * Hkv < 1 << 30:
      return LONE
    if not plan_pays(B, Hkv, width) or resolve_decode_algo(B, Hkv, self.algo) not in (2, 3):
      return None
    return require().decode_plan(ctx_lens, B, Hkv, width, self.Dh)


class PendingMerge:
  """A lone sequence's decode attention in parts whose merge was left to its consumer: o_proj merges what its workgroups multiply in
  its prologue (linear_resid_norm -> gemm_solo_merge), instead of the last workgroup of the attention."""

  __slots__ = ("o", "ml", "ctx_lens", "width", "Hkv", "Dh")

  def __init__(self, o, ml, ctx_lens, width, Hkv, Dh):
    self.o, self.ml, self.ctx_lens, self.width, self.Hkv, self.Dh = o, ml, ctx_lens, width, Hkv, Dh


# Block tables whose parts (2 to 4) the output projection merges: in its prologue they cost it 0.5 us, or 1 us of 8 layers of 4096
# columns, whatever the context; the attention's last workgroup takes 2 to 3 us, but only where there is more than one part.  us a step
# of Llama-3.2-1B / Llama-3-8B (8 layers), left / merged there: 60 tokens 644 / 636 and 835 / 828, 400 664 / 677 and 856 / 862 (8 pages
# both), 600 678 / 687 and 864 / 866, 2000 695 / 699 and 881 / 872
MERGE_PAGES = (9, 16)


def attn_decode(q, k_cache, v_cache, block_tables, ctx_lens, scale: float, ws: DecodeWorkspace | None = None,
                out: torch.Tensor | None = None, defer_merge: bool = False, plan=None):
  """plan: ws.plan of the same step.  defer_merge (plan LONE, MERGE_PAGES wide): return a PendingMerge."""
  if not _gpu(q):
    y = ref.attn_decode(q, k_cache, v_cache, block_tables, ctx_lens, scale)
    if out is not None:
      out.copy_(y.view(out.shape))
      return out
    return y
  B, H, Dh = q.shape
  width = block_tables.shape[1]
  if ws is None:
    ws = DecodeWorkspace(B, H, Dh, width * PAGE, q.device)
  out = torch.empty_like(q) if out is None else out
  if plan is not None:
    nt = B * k_cache.shape[1] * width * PAGE * Dh * 4 >= NT_MIN_KV_BYTES
    lone = plan is LONE
    defer = defer_merge and lone and MERGE_PAGES[0] <= width <= MERGE_PAGES[1]
    require().attn_decode_split(q, k_cache, v_cache, block_tables, None if lone else plan, ctx_lens, ws.tickets, out, ws.o, ws.ml,
                                float(scale), nt, defer)
    return PendingMerge(ws.o, ws.ml, ctx_lens, width, k_cache.shape[1], Dh) if defer else out
  ppp, nparts, algo = ws.partition(B, k_cache.shape[1], width)
  require().attn_decode(q, k_cache, v_cache, block_tables, ctx_lens, out, ws.o, ws.ml, ppp, nparts, float(scale), algo)
  return out


# XOT_PREFILL_ATTN: 2 = 256-row workgroups, LDS-DMA page ring, in-register softmax (default); 1 = the
# first 64-row kernel (register-staged pages, P through LDS)
PREFILL_ALGO = int(os.environ.get("XOT_PREFILL_ATTN", "2"))


def attn_prefill(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, max_qlen: int, scale: float,
                 out: torch.Tensor | None = None) -> torch.Tensor:
  if not _gpu(q):
    y = ref.attn_prefill(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, scale)
    if out is not None:
      out.copy_(y)
      return out
    return y
  out = torch.empty_like(q) if out is None else out
  require().attn_prefill(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, out, int(max_qlen), float(scale),
                         PREFILL_ALGO)
  return out


# ------------------------------------------------------------------ sampling
def attention_bidir(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, B: int, L: int, H: int, Dh: int,
                    scale: float) -> torch.Tensor:
  """Bidirectional (unmasked) multi-head attention over B sequences of L tokens: q / k / v [B*L, H*Dh] token-major
  (row views with unit inner stride) -> o [B*L, H*Dh].  GPU: the flash-style forward of the training kernels with
  the causal mask off (csrc/attention_train.hip; V transposed per head first) for Dh 64 / 128; CPU and other
  head sizes (the tiny test towers): fp32 reference."""
  if not _gpu(q) or Dh not in (64, 128):
    qh, kh, vh = (t.float().reshape(B, L, H, Dh).transpose(1, 2) for t in (q, k, v))
    a = torch.softmax((qh @ kh.transpose(-1, -2)) * scale, -1) @ vh
    return a.transpose(1, 2).reshape(B * L, H * Dh).to(q.dtype)
  C = require()
  Lp = -(-L // 64) * 64
  vt = torch.empty(B, H, Dh, Lp, dtype=v.dtype, device=v.device)
  C.attn_train_transpose(v, vt, B, L, Lp, H, Dh)
  o = torch.empty(B * L, H * Dh, dtype=q.dtype, device=q.device)
  lse2 = torch.empty(B * H * L, dtype=torch.float32, device=q.device)
  C.attn_train_fwd(q, k, vt, o, lse2, B, L, Lp, H, H, Dh, float(scale), False)
  return o


def sample(logits: torch.Tensor, temps: torch.Tensor, top_k: int, seed_off: torch.Tensor,
           out: torch.Tensor | None = None) -> torch.Tensor:
  """Greedy when temp <= 1e-5, else top-k + exponential-race sampling (all on device)."""
  if not _gpu(logits):
    B = logits.shape[0]
    res = torch.empty(B, dtype=torch.int32)
    g = torch.Generator().manual_seed(int(seed_off[0]) * 1000003 + int(seed_off[1]))
    for b in range(B):
      t = float(temps[b])
      row = logits[b].float()
      if t <= 1e-5 or top_k == 1:
        res[b] = int(row.argmax())
        continue
      row = row / max(t, 1e-5)
      if 0 < top_k < row.numel():
        kth = torch.topk(row, top_k).values[-1]
        row = row.masked_fill(row < kth, float("-inf"))
      probs = torch.softmax(row, -1)
      q = torch.empty_like(probs).exponential_(1, generator=g)
      res[b] = int((probs / q).argmax())
    if out is not None:
      out.copy_(res)
      return out
    return res
  out = torch.empty(logits.shape[0], dtype=torch.int32, device=logits.device) if out is None else out
  require().sample(logits, temps, int(top_k), seed_off, out)
  return out


def topk_cand(logits: torch.Tensor, top_k: int, kc: int = 64) -> tuple:
  """Each row's top_k (value, index) candidates in [B, kc] buffers (unused slots -inf / -1): one vocab
  slice's contribution to a sampler that runs on another stage."""
  B = logits.shape[0]
  if not _gpu(logits):
    v, i = torch.topk(logits.float(), top_k, dim=-1)
    vals = torch.full((B, kc), float("-inf"))
    idx = torch.full((B, kc), -1, dtype=torch.int32)
    vals[:, :top_k] = v
    idx[:, :top_k] = i.int()
    return vals, idx
  vals = torch.empty(B, kc, dtype=torch.float32, device=logits.device)
  idx = torch.empty(B, kc, dtype=torch.int32, device=logits.device)
  require().topk_cand(logits, int(top_k), vals, idx)
  return vals, idx


# ------------------------------------------------------------------ DeepSeek MLA
def mla_prep(ckv, kv_ln, q, qpe_off: int, H: int, pos, cos_sin, slots, cache, eps: float) -> None:
  """ckv [T, >= DL+DR] (rows may be strided), q [T, ldq]: latent norm + rope + cache write, q_pe rotated
  in place."""
  if not _gpu(ckv):
    ref.mla_prep(ckv, kv_ln, q, qpe_off, H, pos, cos_sin, slots, cache, eps)
    return
  require().mla_prep(ckv, kv_ln, q, int(qpe_off), int(H), pos, cos_sin, slots, cache, float(eps))


class MLAWorkspace:
  """Split-KV scratch of the MLA attention kernel: ROWS rows of partials a head, which hold the partitions of every step, whatever its
  tokens and its tables' width (128 heads, 512 tokens of up to 32768: 0.13 GB; a bound on the tokens times one on the partitions 6.3)."""

  ROWS = 512  # partition(): tokens x partitions of more than one is below 256 + 255

  def __init__(self, max_tokens: int, H: int, DL: int, max_ctx: int, device):
    self.max_tokens, self.H, self.DL = max_tokens, H, DL
    self.pages = max(1, -(-max_ctx // PAGE))
    self.o = torch.empty(self.ROWS * H * DL, dtype=torch.float32, device=device)
    self.ml = torch.empty(self.ROWS * H * 2, dtype=torch.float32, device=device)

  def wide(self, T: int) -> bool:
    """Many-head kernel (one workgroup covers up to 128 heads, each page loaded once for all of them) for
    >= 64 heads at batch sizes that fill the chip; the narrow kernel (a workgroup per 16 heads) keeps more
    workgroups in flight for a handful of tokens.  XOT_MLA_WIDE=0/1 forces either."""
    force = os.environ.get("XOT_MLA_WIDE")
    if force in ("0", "1"):
      return force == "1"
    return self.H >= 64 and T >= 8

  def partition(self, T: int, width_pages: int):
    """(pages per partition, partitions, wide).  A CU holds one workgroup (two 73 KB pages in LDS): enough for 256 CUs, and not many
    more, since contexts alike fill them all (16 heads, 64 of 900 in tables of 16 pages, us in 4 / 6 parts 24.2 / 31.4, 37 of 900 in 6 / 8
    20.5 / 25.9; but ragged_pages).  Narrow kernel: parts of at least two pages; of one for a
    handful of workgroups on a short table (us in parts of 1 / 2 / 3 / 4 pages, attention and merge: one of 900 9.9 / 11.3 / 13.1 /
    14.8, one of 2000 13.5 / 13.1 / 14.5 / 15.4), but for tables of three and fewer (64 of 100 13.3 in two parts, 9.4 whole).
    More than 128 workgroups on a short table, and those of a prompt's rows (their contexts are alike), stay whole: 16 heads, 200 of up
    to 400 28 in parts of 4 pages, 20.7; 128 heads, 200 new tokens 88 in two parts, 40, behind 2000 243, 199."""
    nhb = -(-self.H // 16)
    wide = self.wide(T)
    units = max(1, T * -(-nhb // 8) if wide else T * nhb)
    want = 1 if units > 128 and (width_pages <= 16 or T > self.max_tokens) else -(-256 // units)
    cap = width_pages if wide or 3 < width_pages <= 16 and units * width_pages <= 128 else width_pages // 2 if width_pages > 3 else 1
    nparts = max(1, min(want, cap))
    ppp = -(-width_pages // nparts)
    return ppp, -(-width_pages // ppp), wide

  def ragged_pages(self, T: int, width_pages: int) -> int:
    """Pages per partition of the narrow kernel for contexts that leave many partitions empty: one and a half workgroups a CU (16 heads,
    37 sequences of 62 .. 867 tokens 15.8 us in partition()'s parts, 14.5 in these, 64 of 65 .. 830 17.5 and 15.9).  Which of the two a
    step of single tokens takes is counted on the device: csrc/mla.hip pages_of_parts."""
    units = T * -(-self.H // 16)
    return -(-width_pages // max(1, min(384 // units, width_pages // 2)))


def mla_attn(q_lat, q_pe, cache, block_tables, cu_q, ctx_lens, scale: float, ws: MLAWorkspace | None = None,
             out: torch.Tensor | None = None) -> torch.Tensor:
  """q_lat [H, T, DL], q_pe [T, >= H*DR] (row-major, strided rows ok) -> o_lat [H, T, DL]."""
  if not _gpu(q_lat):
    y = ref.mla_attn(q_lat, q_pe, cache, block_tables, cu_q, ctx_lens, scale)
    if out is not None:
      out.copy_(y)
      return out
    return y
  H, T, DL = q_lat.shape
  width = block_tables.shape[1]
  if ws is None:
    ws = MLAWorkspace(T, H, DL, width * PAGE, q_lat.device)
  ppp, nparts, wide = ws.partition(T, width)
  even = 0
  if nparts > 1 and not wide and T == ctx_lens.shape[0] <= 64:
    fine = ws.ragged_pages(T, width)
    if fine < ppp:
      even, ppp, nparts = ppp, fine, -(-width // fine)
  out = torch.empty_like(q_lat) if out is None else out
  require().mla_attn(q_lat, q_pe, cache, block_tables, cu_q, ctx_lens, out, ws.o, ws.ml, int(ppp), int(nparts),
                     float(scale), int(wide), int(even))
  return out


_ROUTE_CNT = {}


def _route_counters(device) -> torch.Tensor:
  """Per-device expert counters of moe_route_ds: zero between launches (the kernel resets them)."""
  key = str(device)
  if key not in _ROUTE_CNT:
    _ROUTE_CNT[key] = torch.zeros(256, dtype=torch.int32, device=device)
  return _ROUTE_CNT[key]


def moe_route_ds(logits, bias, k: int, n_group: int, topk_group: int, method: int, sigmoid: bool, norm: bool,
                 scale: float, outs: tuple | None = None):
  """DeepSeekMoE routing.  GPU: (topw, topi, slot_of, sorted_tok, off) device tensors (graph-capturable;
  launches on one stream reuse the per-device counters in order); CPU: (topw [T, k], topi [T, k])."""
  if not _gpu(logits):
    return ref.moe_route_ds(logits, bias, k, n_group, topk_group, method, sigmoid, norm, scale)
  T, E = logits.shape
  dev = logits.device
  if outs is None:
    outs = (torch.empty(T * k, dtype=torch.float32, device=dev), torch.empty(T * k, dtype=torch.int32, device=dev),
            torch.empty(T * k, dtype=torch.int32, device=dev), torch.empty(T * k, dtype=torch.int32, device=dev),
            torch.empty(E + 1, dtype=torch.int32, device=dev))
  require().moe_route_ds(logits.contiguous(), bias, int(k), int(n_group), int(topk_group), int(method), bool(sigmoid),
                         bool(norm), float(scale), _route_counters(dev), *outs)
  return outs


# ------------------------------------------------------------------ mixers on an fp32 residual stream (csrc/mixers.hip)
# P is a fused projection's fp32 output [T, n]; *_off are column offsets into it.  Outputs are preallocated by the
# caller (graph-capturable); activation outputs may be column slices of a wider row buffer.
def _mix(name: str, on_gpu: bool):
  return getattr(require(), name) if on_gpu else getattr(ref, name)


def resid_scale_norm(x, y1=None, s1=None, y2=None, s2=None, gain=None, eps: float = 1e-5, out=None) -> None:
  """fp32 residual rows x [T, D] += s1 * y1 (+ s2 * y2) in place (per-channel scales; y rows may be wider than
  D), then, with `out`, out[:, :D] = x / sqrt(mean(x^2) + eps) * gain (gain: one fp32 number on the device)."""
  _mix("resid_scale_norm", _gpu(x))(x, y1, s1, y2, s2, gain, float(eps), out)


def embed_rows(ids, table, want_ids: bool = False):
  """(rows of the fp32 table [V, D] at ids [T] clamped to it, the clamped ids as int32 or None)."""
  if not (_gpu(table) and table.dtype == torch.float32 and ids.dtype in (torch.int32, torch.int64)):
    ids = ids.long().clamp(0, table.shape[0] - 1)
    return table.index_select(0, ids), ids.to(torch.int32) if want_ids else None
  h = torch.empty(ids.numel(), table.shape[1], dtype=table.dtype, device=table.device)
  ids32 = torch.empty(ids.numel(), dtype=torch.int32, device=table.device) if want_ids else None
  require().embed_rows(ids.contiguous(), table, h, ids32)
  return h, ids32


def gelu_mul(P, gate_off: int, up_off: int, F: int, out) -> None:
  """out[:, :F] = gelu_tanh(P[:, gate_off : +F]) * P[:, up_off : +F]  (out rows may be wider: K padding).  up_off -1: gate and
  up columns alternate in tiles of 16 from gate_off on."""
  _mix("gelu_mul", _gpu(P))(P, int(gate_off), int(up_off), int(F), out)


def rope_kv_store(P, q_off: int, k_off: int, v_off: int, H: int, G: int, d: int, R: int, pos, cos_sin, slots, q_out,
                  k_cache, v_cache) -> None:
  """Rotate-half RoPE on the first R dims of every q / k head (pairs (i, i + R/2)); q -> q_out [T, H, d], the
  rotated key -> k_cache [pages, G, 64, d], the value (v_off < 0: the key before rotation) -> v_cache [pages, G, d, 64],
  both at `slots`."""
  qk_norm_rope_store(P, None, q_off, k_off, k_off if v_off < 0 else v_off, H, G, d, d, R, pos, cos_sin, slots, 0.0, False, q_out,
                     k_cache, v_cache)


def attn_gated_chunk(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, pb, scale: float, chunk: int, out_scale: float,
                     out, max_qlen: int = 0) -> None:
  """out [T, H d] = out_scale * sum over the keys j <= i of query i's chunk (floor(i / chunk) == floor(j / chunk))
  of sigmoid(q_i . k_j * scale + pb[head]) v_j; positions count from each sequence's start.  Caches: K [pages, G, 64,
  d], V [pages, G, d, 64].  max_qlen: the step's longest run of new tokens of one sequence (0: unknown -> the total);
  bf16 steps with runs above one token take the MFMA kernel; single tokens, fp32 and head sizes that are no
  multiple of 32 a (token, kv head, key split) kernel that scores each key once for all query heads of its group."""
  _mix("attn_gated_chunk", _gpu(q))(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, pb, float(scale), int(chunk),
                                    float(out_scale), out, int(max_qlen) or int(q.shape[0]))


def delta_prep(P, x_off: int, b_off: int, a_off: int, conv_w, conv_state, state_slots, cu_q, A_log, dt_bias, H: int,
               G: int, d: int, dv: int, qkv, beta, decay) -> None:
  """Delta-rule inputs of a step and the convolution state's update: channels [q: G d | k: G d | v: H dv] at P[:, x_off ...];
  q = unit(silu(conv q)) d^-1/2, k = unit(silu(conv k)), v = silu(conv v) -> qkv [T, C]; beta and decay: delta_gates.  (A model
  step calls conv_prep with the units that its weights hold on the device.)"""
  units, width = ref.conv_units(ref.delta_units(H, G, d, dv), conv_w.shape[0])
  conv_prep(P, x_off, conv_w, None, units.to(P.device), None, conv_state, state_slots, cu_q, 0.0, qkv.view(P.shape[-2], conv_w.shape[0]),
            width=width, delta=(b_off, a_off, dt_bias, A_log, beta, decay))


def gla_prep(P, a1_off: int, a2, a2_b, tau: float, decay) -> None:
  """decay [T, H d] = sigmoid(z)^(1/tau), z = a2 P[:, a1_off : +rank] + a2_b."""
  _mix("gla_prep", _gpu(P))(P, int(a1_off), a2, a2_b, float(tau), decay)


conv_units = ref.conv_units


def conv_prep(P, x_off: int, conv_w, conv_b, units, norm_w, conv_state, state_slots, cu_q, eps: float, out, max_qlen: int = 0,
              width: int = 256, gates: tuple | None = None, steps: tuple | None = None, delta: tuple | None = None) -> None:
  """Causal convolutions over time of the channels P[:, x_off : +C] (conv_w [C, taps], last column the current token; conv_b
  [C] or None) -> out [T, C] fp32, then per unit (conv_units) SiLU and a unit length or a weighted RMS norm (norm_w).  The
  inputs before the step come from conv_state [slots, taps - 1, C], which takes the step's last ones.  max_qlen 1: every
  sequence has one new token (the state is updated in the same launch).  width: the most channels of a unit.  P may be [T, n]
  or unreduced split-K slabs [S, T, n] (also below).  gates / steps / delta: the arguments behind P of recurrence_gates,
  ssd_steps or delta_gates, which read the same projection: done as well, for single tokens in the same launch."""
  if _gpu(P) and max_qlen == 1 and P.shape[-2] == state_slots.numel() and sum(g is not None for g in (gates, steps, delta)) == 1:
    if delta is not None:
      b_off, dt_off, dt_bias, A_log, beta, decay = delta
      a1_off = g1_off = 0
      a2 = g2 = gate = dt = None
    elif gates is not None:
      b_off, beta, a1_off, a2, dt_bias, A_log, decay, g1_off, g2, gate = gates
      dt_off, dt = 0, None
    else:
      dt_off, dt_bias, A_log, dt, decay = steps
      b_off = a1_off = g1_off = 0
      beta = a2 = g2 = gate = None
    require().conv_prep_gates(P, int(x_off), conv_w, conv_b, units, norm_w, conv_state, state_slots, cu_q, float(eps), out, int(width),
                              int(b_off), beta, int(a1_off), a2, dt_bias, A_log, decay, int(g1_off), g2, gate, int(dt_off), dt)
    return
  _mix("conv_prep", _gpu(P))(P, int(x_off), conv_w, conv_b, units, norm_w, conv_state, state_slots, cu_q, float(eps), out,
                             int(max_qlen), int(width))
  if gates is not None:
    recurrence_gates(P, *gates)
  if steps is not None:
    ssd_steps(P, *steps)
  if delta is not None:
    delta_gates(P, *delta)


def delta_gates(P, b_off: int, a_off: int, dt_bias, A_log, beta, decay) -> None:
  """beta [T, H] = sigmoid(P[:, b_off : +H]), decay [T, H] = exp(-exp(A_log) softplus(P[:, a_off : +H] + dt_bias))."""
  _mix("delta_gates", _gpu(P))(P, int(b_off), int(a_off), dt_bias, A_log, beta, decay)


def recurrence_gates(P, b_off: int, beta, a1_off: int, a2, dt_bias, A_log, decay, g1_off: int, g2, gate, za=None) -> None:
  """Gates of the channel-decay delta rule: beta [T, H] = sigmoid(P[:, b_off : +H]); decay [T, H d] = exp(-exp(A_log[head])
  softplus(a2 P[:, a1_off : +rank] + dt_bias)) (za [T, >= H d]: that product, already made); gate [T, H dv] (or None) =
  g2 P[:, g1_off : +rank], without its sigmoid."""
  _mix("recurrence_gates", _gpu(P))(P, int(b_off), beta, int(a1_off), a2, dt_bias, A_log, decay, int(g1_off), g2, gate, za)


def ssd_steps(P, dt_off: int, dt_bias, A_log, dt, decay) -> None:
  """dt [T, H] = softplus(P[:, dt_off : +H] + dt_bias), decay [T, H] = exp(-exp(A_log) dt)."""
  _mix("ssd_steps", _gpu(P))(P, int(dt_off), dt_bias, A_log, dt, decay)


def linear_recurrence(q, k, v, decay, beta, q_scale: float, state, state_slots, cu_q, out, plain: bool = False,
                      max_qlen: int = 0) -> None:
  """Per sequence and value head, token by token on the fp32 state, stored S^T [slots, H, dv, d] (updated in place):
  beta given (delta rule, decay [T, H], or [T, H d] per key channel):  S *= g; u = beta (v - S^T k); S += k u^T; o = S^T q
  (plain: beta scales the input of the plain write instead, S = g S + k (beta v)^T)
  else (decay [T, H d] per key channel, [T, H] per head, or a 1-D [H]: fixed per head):  S = diag(a) S + k v^T; o = S^T q.
  q is scaled by q_scale.
  A state with one value channel more than v has (decay [T, H], beta [T, H] an input scale): S = g S + k (beta [v | 1])^T,
  the last channel being a normaliser n = g n + beta k; out [T, H (dv + 1)] then ends each head with n . q.
  max_qlen: tokens of the step's longest sequence (0: not known); long ones run in chunks of 16 tokens on the GPU."""
  if _gpu(q):
    require().linear_recurrence(q, k, v, decay, beta, float(q_scale), state, state_slots, cu_q, out, bool(plain), int(max_qlen))
  else:
    ref.linear_recurrence(q, k, v, decay, beta, float(q_scale), state, state_slots, cu_q, out, bool(plain))


def gated_rmsnorm(o, w, P, g_off: int, eps: float, out_scale: float, out) -> None:
  """out [T, H dv] = o / rms(o per head) * w * silu(P[:, g_off : +H dv]) * out_scale."""
  _mix("gated_rmsnorm", _gpu(o))(o, w, P, int(g_off), float(eps), float(out_scale), out)


def recurrence_norm(q, k, v, decay, beta, q_scale: float, state, state_slots, cu_q, w, gate, sigmoid: bool, eps: float, scale: float,
                    out, gla=None, max_qlen: int = 0, gelu=None, chan=None) -> None:
  """linear_recurrence, then each head's RMS norm times w ([dv], or one per head [H dv]), gate [T, H dv]'s silu (or its logistic
  function) and scale -> out [T, >= H dv].  gla: (P, first column, a2, a2_b, tau) of gla_prep, which then makes the decays.  gelu:
  arguments of a gelu_mul that is done along with it.  chan: (P, column of the step sizes, za, dt_bias, A_log) of recurrence_gates, which
  then makes decays and write strengths.  A step of single tokens is one launch on the GPU (csrc/recurrence_step.hip)
  where that covers the sizes; prompts' decays are made inside the recurrence (csrc/recurrence_chunk.hip) where it takes them."""
  def made_gates():
    P, b_off, za, dt_bias, A_log = chan
    beta = torch.empty(q.shape[0], A_log.numel(), dtype=torch.float32, device=q.device)
    decay = torch.empty(q.shape[0], dt_bias.numel(), dtype=torch.float32, device=q.device)
    recurrence_gates(P, b_off, beta, 0, None, dt_bias, A_log, decay, 0, None, None, za=za)
    return decay, beta
  apart = 0 < max_qlen < 32 or not _gpu(q)  # (never by chunks: 1.2 us less of the host's time than asking)
  if chan is not None and apart:
    decay, beta = made_gates()
    chan = None
  if max_qlen == 1 and _gpu(q):
    a1, a2, a2_b, tau = (gla[0][:, gla[1]:gla[1] + gla[2].shape[1]], *gla[2:]) if gla is not None else (None, None, None, 0.0)
    for g in ((gelu, None) if gelu is not None else (None,)):  # (an activation it cannot take along has a launch of its own)
      if require().recurrence_step(q, k, v, decay, beta, float(q_scale), state, state_slots, cu_q, a1, a2, a2_b, float(tau), w, gate,
                                   bool(sigmoid), float(eps), float(scale), out, *(g or (None, 0, 0, 0, None))):
        if gelu is not None and g is None:
          gelu_mul(*gelu)
        return
  if gelu is not None:
    gelu_mul(*gelu)
  T, H, dv, d = q.shape[0], state.shape[1], state.shape[2], state.shape[3]
  o = torch.empty(T, H * dv, dtype=torch.float32, device=q.device)
  done = False
  if chan is not None:
    P, b_off, za, dt_bias, A_log = chan
    done = require().linear_recurrence_made(q, k, v, P, int(b_off), za, dt_bias, 1.0, A_log, float(q_scale), state, state_slots, cu_q, o, int(max_qlen))
    if not done:
      decay, beta = made_gates()
  elif gla is not None:
    # A chunk's low-rank product is a chain of its own, tile by tile, which pays from a quarter of a (chunk, head) a SIMD on, at key
    # dims of 128 from one; us a launch of its own / made by the chunks, rank 16: 4 heads of 64, one of 300 tokens 21.8 / 23.7, of 1000 49.1 /
    # 48.2, 16 heads of 1000 53 / 50, 12 of 1000 206 / 187; 16 heads of 128, one of 300 29.6 / 34.3, of 1000 65.4 / 63.6, 12 of 1000 346 / 325.
    waves = (T // 16 + state_slots.numel()) * H
    if not apart and beta is None and gla[0].dim() == 2 and waves >= (256 if d == 64 else 1024):
      P, a1_off, a2, a2_b, tau = gla
      done = require().linear_recurrence_made(q, k, v, P, int(a1_off), a2, a2_b, float(tau), None, float(q_scale), state, state_slots, cu_q, o, int(max_qlen))
    if not done:
      decay = torch.empty(T, H * d, dtype=torch.float32, device=q.device)
      gla_prep(*gla, decay)
  if not done:
    linear_recurrence(q, k, v, decay, beta, q_scale, state, state_slots, cu_q, o, max_qlen=max_qlen)
  if sigmoid:  # (that pass has a weight per head and no scale)
    wh = w if w.numel() == H * dv else w.repeat(H)
    gated_group_norm(o, None, wh if scale == 1.0 else wh * scale, gate, 0, H, eps, out)
  elif w.numel() == dv:
    gated_rmsnorm(o, w, gate, 0, eps, scale, out[:, :H * dv])
  else:  # (that one has a weight for all heads)
    y = torch.empty_like(o)
    gated_rmsnorm(o, torch.ones_like(w[:dv]), gate, 0, eps, scale, y)
    out[:, :H * dv].copy_(y * w)


# ------------------------------------------------------------------ post-norm blocks (csrc/hybrid.hip)
pool_dims = ref.pool_dims


def gated_postnorm(x, y, P, g_off: int, gate_b, alpha: float, w, eps: float, out=None) -> None:
  """fp32 stream rows x [T, D] <- (alpha x + y * sigmoid(P[:, g_off : +D] + gate_b)) / rms * w in place (P None: the
  sublayer's result y is not gated); with `out`, out[:, :D] = the new x in out's dtype (the next GEMM's operand)."""
  _mix("gated_postnorm", _gpu(x))(x, y, P, int(g_off), gate_b, float(alpha), w, float(eps), out)


def qk_norm_rope_store(P, bias, q_off: int, k_off: int, v_off: int, H: int, G: int, d: int, dv: int, R: int, pos, cos_sin,
                       slots, eps: float, qk_norm: bool, q_out, k_cache, v_cache, q_norm=None, k_norm=None) -> None:
  """q / k / v = P's columns (+ bias, one fp32 number per column of P); with q_norm [H d] (and k_norm [G d] for the keys)
  all of a token's q numbers together are divided by their RMS and weighted (the keys likewise); rotate-half RoPE on the
  first R dims of every q / k head, then (qk_norm) each head divided by its RMS; q -> q_out [T, H, d], k -> k_cache [pages, G, 64, d],
  v -> v_cache [pages, Gv, dv, 64] at `slots` (Gv = v_cache's heads: G, or fewer when neighbouring key heads share a
  value head).  k_off < 0: the layer has no keys and values of its own."""
  _mix("qk_norm_rope_store", _gpu(P))(P, bias, int(q_off), int(k_off), int(v_off), int(H), int(G), int(d), int(dv), int(R),
                                      pos, cos_sin, slots, float(eps), bool(qk_norm), q_out, k_cache, v_cache, q_norm, k_norm)


def kv_pool_update(k_cache, v_cache, kp, vp, block_tables, cu_q, ctx_lens, pool: int, max_qlen: int) -> None:
  """Mean key and value of every block of `pool` consecutive tokens whose last token is among the step's new ones,
  read from the paged caches as they hold them, into the pooled caches kp [pages, G, per, d] / vp [pages, G, per, dv]
  (entry of block b: with the page of its last token, see pool_dims)."""
  _mix("kv_pool_update", _gpu(k_cache))(k_cache, v_cache, kp, vp, block_tables, cu_q, ctx_lens, int(pool), int(max_qlen))


def attn_window_pool(q, k_cache, v_cache, kp, vp, block_tables, cu_q, ctx_lens, sink, scale: float, window: int,
                     pool: int, out, max_qlen: int = 0, chunk: int = 0, keep: int = 0, softcap: float = 0.0) -> None:
  """out [T, H dv] = softmax attention of each new token over the tokens at most window - 1 places back (window 0:
  all) and, with chunk > 0, in its own block of `chunk` positions (counted from the sequence's start), the sequence's first
  `keep` tokens wherever the query is (no pooled blocks then), the pooled blocks that end at or before position - window (pool 0: none), and the per-head sink logit.  Key
  head g reads value head g / (G / Gv) (the caches' head counts); out may be fp32 beside bf16 caches.  softcap > 0:
  scores are softcap * tanh(score / softcap)."""
  _mix("attn_window_pool", _gpu(q))(q, k_cache, v_cache, kp, vp, block_tables, cu_q, ctx_lens, sink, float(scale),
                                    int(window), int(pool), out, int(max_qlen) or int(q.shape[0]), int(chunk), int(keep),
                                    float(softcap))


def ssd_prep(P, x_off: int, dt_off: int, conv_w, conv_b, conv_state, state_slots, cu_q, A_log, dt_bias, H: int, dv: int,
             xbc, v, decay) -> None:
  """SSD inputs of a step: xbc [T, C] = silu(causal conv of P[:, x_off : +C] + conv_b) (x | B | C channels),
  dt = softplus(P[:, dt_off : +H] + dt_bias), v [T, H dv] = dt * x, decay [T, H] = exp(-exp(A_log) dt); the
  convolution state [slots, taps - 1, C] takes the step's last inputs."""
  _mix("ssd_prep", _gpu(P))(P, int(x_off), int(dt_off), conv_w, conv_b, conv_state, state_slots, cu_q, A_log, dt_bias,
                            int(H), int(dv), xbc, v, decay)


def ssd_gate_norm(o, xbc, skip_d, P, z_off: int, w, groups: int, eps: float, out) -> None:
  """out[:, :inner] = group_rms_norm((o + D[head] * x) * silu(P[:, z_off : +inner])) * w, in `groups` equal parts."""
  _mix("ssd_gate_norm", _gpu(o))(o, xbc, skip_d, P, int(z_off), w, int(groups), float(eps), out)


def polynorm_act(P, up_off: int, F: int, coef, eps: float, out) -> None:
  """out[:, :F] = a N(z) + b N(z^2) + c N(z^3) + e, z = P[:, up_off : +F], N = division by the row's RMS, coef = (a, b, c, e)."""
  _mix("polynorm_act", _gpu(P))(P, int(up_off), int(F), coef, float(eps), out)


def relu2(P, off: int, F: int, out) -> None:
  """out[:, :F] = relu(P[:, off : +F])^2."""
  _mix("relu2", _gpu(P))(P, int(off), int(F), out)


def moe_weighted_sum(y, slot_of, topw, k: int, sh_y, P, shg_off: int, out, splits: int = 1) -> None:
  """out [T, D] fp32 = sum_j topw[t, j] * y[slot_of[t, j]] (+ sigmoid(P[t, shg_off]) * sh_y[t] for a shared expert);
  y [splits * T k, >= D]: the experts' down projections, K slice after K slice."""
  _mix("moe_weighted_sum", _gpu(y))(y, slot_of, topw, int(k), sh_y, P, int(shg_off), out, int(splits))


# ------------------------------------------------------------------ sandwich blocks (csrc/latent.hip)
def sandwich_add_norm(x, y, wb, wn, eps: float, out=None, bb=None, bn=None, mult: float = 1.0, yb=None, layer: bool = False) -> None:
  """fp32 stream rows x [T, D] += mult * norm(y + yb) * wb in place (y None: nothing is added; yb: one fp32 number per
  column, or None); with wn, out[:, :D] = norm(x) * wn in out's dtype (the next GEMM's operand), with out alone out[:, :D] =
  x.  norm = division by the RMS, or, with the biases bb / bn or
  with `layer`, the layer norm (v - mean) / sqrt(var + eps) * w (+ b)."""
  _mix("sandwich_add_norm", _gpu(x))(x, y, wb, wn, float(eps), out, bb, bn, float(mult), yb, bool(layer))


def latent_kv_store(P, ckv_off: int, R: int, dr: int, kv_norm, q_off: int, q_rank: int, q_norm, eps: float, rot_dims: int,
                    interleaved: bool, pos, cos_sin, slots, cache, qa_out) -> None:
  """Per token: the latent rms_norm(P[:, ckv_off : +R]) * kv_norm and the rotated key part rope(P[:, ckv_off + R : +dr])
  -> cache [pages, 1, 64, R + dr] at `slots`; q_rank > 0: qa_out[:, :q_rank] = rms_norm(P[:, q_off : +q_rank]) * q_norm
  (the query latent, operand of the query up-projection).  RoPE on the first rot_dims dims of the rotated part, pairs
  (2i, 2i + 1) (interleaved) or (i, i + rot_dims / 2); cos_sin [rows, rot_dims] = (cos | sin)."""
  _mix("latent_kv_store", _gpu(P))(P, int(ckv_off), int(R), int(dr), kv_norm, int(q_off), int(q_rank), q_norm, float(eps),
                                   int(rot_dims), bool(interleaved), pos, cos_sin, slots, cache, qa_out)


def latent_q_rope(Q, q_off: int, H: int, dn: int, dr: int, rot_dims: int, interleaved: bool, pos, cos_sin, qn_out,
                  qpe_out) -> None:
  """Queries Q[:, q_off : +H (dn + dr)], head by head [dn unrotated | dr rotated]: the unrotated parts -> qn_out
  [H, T, dn] (operand of the per-head product with W_uk), the rotated parts after RoPE -> qpe_out [T, H, dr]."""
  _mix("latent_q_rope", _gpu(Q))(Q, int(q_off), int(H), int(dn), int(dr), int(rot_dims), bool(interleaved), pos, cos_sin,
                                 qn_out, qpe_out)


def latent_attn(q_lat, q_pe, cache, block_tables, cu_q, ctx_lens, sink, scale: float, window: int, out,
                max_qlen: int = 0) -> None:
  """out [H, T, R] = softmax attention of every head's absorbed query (q_lat [H, T, R] against the cached latents, q_pe
  [T, H, dr] against the cached rotated key parts, times scale) over the tokens at most window - 1 places back
  (window 0: all earlier ones), the values being the latents themselves; sink [H] (or None): one more logit per head in
  the denominator.  cache [pages, 1, 64, R + dr]."""
  _mix("latent_attn", _gpu(q_lat))(q_lat, q_pe, cache, block_tables, cu_q, ctx_lens, sink, float(scale), int(window), out,
                                   int(max_qlen) or int(q_lat.shape[1]))


def latent_out_gate(o, P, g_off: int, gate: int, out) -> None:
  """o [H, T, dv] -> out[:, :H dv] (token-major, out's dtype) times sigmoid(P[:, g_off : ...]): gate 0 none, 1 one
  gate per element, 2 one per head."""
  _mix("latent_out_gate", _gpu(o))(o, P, int(g_off), int(gate), out)


def glu_act(P, gate_off: int, up_off: int, F: int, clamped: bool, limit: float, out) -> None:
  """out[:, :F] = silu(g) * u, or (clamped) g' sigmoid(1.702 g') (u' + 1) with g' = min(g, limit), u' = clamp(u,
  -limit, limit); g = P[:, gate_off : +F], u = P[:, up_off : +F]."""
  _mix("glu_act", _gpu(P))(P, int(gate_off), int(up_off), int(F), bool(clamped), float(limit), out)


def gelu_gather_mul(P, off: int, table, ids, col0: int, n: int, out) -> None:
  """out[:, :n] = gelu_tanh(P[:, off : +n]) * table[ids, col0 : +n]; table [V, cols] in out's dtype, ids [T] int32 (rows of
  the table; ids outside it are clamped)."""
  _mix("gelu_gather_mul", _gpu(P))(P, int(off), table, ids, int(col0), int(n), out)


# ------------------------------------------------------------------ layer-norm sandwich blocks (csrc/recurrent_gates.hip)
def diff_attn_out(a, P, g_off: int, H: int, G: int, lam: float, post: float, eps: float, out) -> None:
  """Differential attention's combination: a [T, 2 H dv] fp32, the two maps' outputs with heads ordered (kv head, map, head
  of the group) -> out[:, :H dv] = rms_norm(a_1 - lam a_2) * post * sigmoid(P[:, g_off + head])."""
  _mix("diff_attn_out", _gpu(a))(a, P, int(g_off), int(H), int(G), float(lam), float(post), float(eps), out)


def sigmoid_gate_mul(a, P, g_off: int, out) -> None:
  """out[:, :n] = a * sigmoid(P[:, g_off : +n]) for a [T, n], fp32 or of out's dtype (out's own rows: in place)."""
  _mix("sigmoid_gate_mul", _gpu(a))(a, P, int(g_off), out)


def silu_cols(P, off: int, n: int, out) -> None:
  """out [T, n] fp32 = silu(P[:, off : +n])."""
  _mix("silu_cols", _gpu(P))(P, int(off), int(n), out)


def mlstm_gates(P, i_off: int, f_off: int, gate_b, cap: float, mstate, state_slots, cu_q, decay, inscale, mout) -> None:
  """The mlstm's gates of a step, per head: i = cap tanh((P[i_off + h] + gate_b[h]) / cap), f = logsigmoid(cap tanh((P[f_off
  + h] + gate_b[H + h]) / cap)), the running maximum m_t = max(f + m_(t-1), i) continued from mstate [slots, H] (updated
  in place); decay [T, H] = e^(f + m_(t-1) - m_t), inscale = e^(i - m_t), mout = m_t."""
  _mix("mlstm_gates", _gpu(P))(P, int(i_off), int(f_off), gate_b, float(cap), mstate, state_slots, cu_q, decay, inscale, mout)


def gated_group_norm(o, m, w, P, g_off: int, groups: int, eps: float, out) -> None:
  """out[:, :groups gs] = o's values divided by their group's RMS, times w, times sigmoid(P[:, g_off : ...]).  With m
  [T, groups] every group of o carries one channel more, a normaliser n, and its values are first divided by max(|n|,
  e^(-m)) + 1e-6."""
  _mix("gated_group_norm", _gpu(o))(o, m, w, P, int(g_off), int(groups), float(eps), out)


def pair_norm_mean(y1, y2, w, eps: float, out) -> None:
  """out [T, D] fp32 = (rms_norm(y1) * w[0] + rms_norm(y2) * w[1]) / 2."""
  _mix("pair_norm_mean", _gpu(y1))(y1, y2, w, float(eps), out)
