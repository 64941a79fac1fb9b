"""Grouped expert GEMMs (csrc/gemm_group.hip and the grouped order of csrc/gemm_big.hip): experts without rows, row counts at the
edges of every row tile, K slices, gathered rows, and the rule that picks a kernel."""
import os
import subprocess
import sys

import pytest
import torch

from xotorch_support_jetson_amd.models.transformer import moe_tiles
from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops.weights_layout import shuffle_for_stream

COUNTS = {
  5: [0, 1, 300, 0, 129],
  17: [0, 1, 0, 15, 16, 17, 31, 32, 33, 0, 48, 49, 64, 65, 130, 200, 2],
}


def integers(gen, *shape):
  return torch.randint(-3, 4, shape, generator=gen).to(torch.bfloat16)


def experts(E, N, Kd, gpu):
  """Integer rows and weights of E experts; (x of fewer rows, x by slot, offsets, gather, shuffled weights, exact products)."""
  g = torch.Generator().manual_seed(E + N + Kd)
  counts = COUNTS[E]
  slots, T = sum(counts), max(counts)
  x, w = integers(g, T, Kd), integers(g, E, N, Kd)
  tok = torch.cat([torch.randperm(T, generator=g)[:n] for n in counts]).int()
  off = torch.tensor([0] + counts).cumsum(0).int()
  xs = x[tok.long()]
  full = torch.cat([xs[off[e]:off[e + 1]].float() @ w[e].float().t() for e in range(E)])
  wide = torch.zeros(T, Kd + 16, dtype=torch.bfloat16, device=gpu)
  wide[:, 8:8 + Kd] = x.to(gpu)
  ws = torch.stack([shuffle_for_stream(m.to(gpu)) for m in w])
  return wide[:, 8:8 + Kd], xs.to(gpu), off.to(gpu), tok.to(gpu), ws, full, slots, T


def test_rule():
  """Streamed where the expert weights are all there is to read; tiles by the rows an expert has."""
  assert moe_tiles(64, 2, 8) == moe_tiles(37, 6, 64) == moe_tiles(340, 6, 64) == moe_tiles(65, 1, 8) == (0, 0, 0)
  assert moe_tiles(65, 2, 8) == moe_tiles(384, 2, 8) == moe_tiles(48, 2, 4) == (1128, 1128, 2)
  assert moe_tiles(342, 6, 64) == moe_tiles(1024, 6, 64) == (2128, 2128, 2)
  assert moe_tiles(385, 2, 8) == (192, 192, 4) and moe_tiles(8192, 6, 64) == (256, 256, 2)


@pytest.mark.parametrize("rows,tiled", [("8", [True] * 4), ("60", [False] * 3 + [True])])
def test_switch_moves_every_line(rows, tiled):
  """XOT_MOE_BIG_MIN_ROWS: one line for few and for many experts, steps of up to 64 tokens included (8, 12, 16 and 64 rows)."""
  code = ("from xotorch_support_jetson_amd.models.transformer import moe_tiles\n"
          "print([moe_tiles(*a)[0] > 0 for a in ((32, 2, 8), (128, 6, 64), (64, 2, 8), (256, 2, 8))])")
  got = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, XOT_MOE_BIG_MIN_ROWS=rows), capture_output=True, text=True, check=True)
  assert got.stdout.strip() == str(tiled)


@pytest.mark.gpu
@pytest.mark.parametrize("E,bm", [(17, 0), (5, 0), (17, 1128), (5, 1128), (17, 2128), (5, 2256)])
@pytest.mark.parametrize("N,Kd,S", [(256, 128, 1), (512, 1408, 1), (256, 1024, 4), (4352, 768, 2)])
def test_experts_exact(gpu, E, bm, N, Kd, S):
  """Integer operands: fp32 sums bit for bit (K slices added here), gathered from a wider buffer and by slot; no row that is not an
  expert's is written.  4352 columns in two slices: the experts follow one another in the tile kernels, else they advance together."""
  from xotorch_support_jetson_amd.ops._ext import require
  C = require()
  x, xs, off, tok, ws, full, slots, T = experts(E, N, Kd, gpu)
  for src, gather in ((x, tok), (xs, None)):
    y = torch.full((S * slots, N), 7.0, device=gpu)
    C.gemm_moe(src, ws, y, off, gather, K.EPI["none"], T, True, S, bm)
    assert torch.equal(y.view(S, slots, N).sum(0).cpu(), full)


@pytest.mark.gpu
@pytest.mark.parametrize("E", [17, 5])
def test_group_epilogues(gpu, E):
  """bf16 results and gated pairs (2^-8 of the value: one rounding; the exponential's error is far below)."""
  from xotorch_support_jetson_amd.ops._ext import require
  C = require()
  N, Kd = 384, 640
  x, _, off, tok, ws, full, slots, T = experts(E, N, Kd, gpu)
  y = torch.empty(slots, N, dtype=torch.bfloat16, device=gpu)
  C.gemm_moe(x, ws, y, off, tok, K.EPI["none"], T, True, 1, 0)
  torch.testing.assert_close(y.cpu().float(), full, rtol=2 ** -8, atol=0)
  gate, up = (full.double().view(slots, N // 32, 2, 16)[:, :, i].reshape(slots, -1) for i in (0, 1))
  a = torch.empty(slots, N // 2, dtype=torch.bfloat16, device=gpu)
  C.gemm_moe(x, ws, a, off, tok, K.EPI["silu"], T, True, 1, 0)
  torch.testing.assert_close(a.cpu().double(), gate * torch.sigmoid(gate) * up, rtol=2 ** -7, atol=1e-6)
  C.gemm_moe(x, ws, a, off, tok, K.EPI["clamp_glu"], T, True, 1, 0, 7.0)
  gc, uc = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
  torch.testing.assert_close(a.cpu().double(), gc * torch.sigmoid(1.702 * gc) * (uc + 1), rtol=2 ** -7, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 16, 64, 65, 150])
@pytest.mark.parametrize("n", [1, 2])
@pytest.mark.parametrize("N,Kd,S", [(256, 128, 1), (128, 1408, 1), (384, 1024, 4)])
def test_shared_experts_exact(gpu, T, n, N, Kd, S):
  """Shared experts of every token behind the routed ones: matrices of n N rows and of n K columns, bit for bit on integers, and
  their rows in the combine (bf16 of an fp32 sum: one rounding)."""
  from xotorch_support_jetson_amd.ops._ext import require
  C = require()
  g = torch.Generator().manual_seed(T + n + N)
  E, k = 17, 2
  x, w, wr, wc = integers(g, T, Kd), integers(g, E, N, Kd), integers(g, n * N, Kd), integers(g, N, n * Kd)
  topi = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
  order = torch.argsort(topi.reshape(-1), stable=True)
  off = torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(topi.reshape(-1), minlength=E).cumsum(0)]).int()
  tok, routed, slots = (order // k).int(), T * k, T * (k + n)
  ws = torch.stack([shuffle_for_stream(m.to(gpu)) for m in w])
  shr, shc = shuffle_for_stream(wr.to(gpu)), shuffle_for_stream(wc.to(gpu))
  full = torch.cat([x[tok[off[e]:off[e + 1]].long()].float() @ w[e].float().t() for e in range(E)])
  y = torch.full((S * slots, N), 7.0, device=gpu)
  C.gemm_moe(x.to(gpu), ws, y, off.to(gpu), tok.to(gpu), K.EPI["none"], T, True, S, 0, w_sh=shr)
  got = y.view(S, slots, N).sum(0).cpu()
  assert torch.equal(got[:routed], full)
  assert torch.equal(got[routed:], torch.cat([x.float() @ wr[j * N:(j + 1) * N].float().t() for j in range(n)]))
  xs = torch.cat([x[tok.long()], integers(g, n * T, Kd)])
  C.gemm_moe(xs.to(gpu), ws, y, off.to(gpu), None, K.EPI["none"], T, True, S, 0, w_sh=shc)
  sh = torch.cat([xs[routed + j * T:routed + (j + 1) * T].float() @ wc[:, j * Kd:(j + 1) * Kd].float().t() for j in range(n)])
  got = y.view(S, slots, N).sum(0).cpu()
  assert torch.equal(got[:routed], full) and torch.equal(got[routed:], sh)
  topw, h = torch.rand(T * k, generator=g), torch.randn(T, N, generator=g).to(torch.bfloat16)
  slot_of = torch.empty(T * k, dtype=torch.int32)
  slot_of[order] = torch.arange(T * k, dtype=torch.int32)
  want = h.double() + sum(sh.double().view(n, T, N)) + (topw.double()[:, None] * full.double()[slot_of.long()]).view(T, k, N).sum(1)
  out = h.to(gpu)
  C.moe_combine(y, slot_of.to(gpu), topw.to(gpu), out, S, n)
  torch.testing.assert_close(out.cpu().double(), want, rtol=2 ** -8, atol=1e-3)
  h2, normed = h.to(gpu), torch.empty(T, N, dtype=torch.bfloat16, device=gpu)
  C.moe_combine_norm(y, slot_of.to(gpu), topw.to(gpu), h2, S, torch.ones(N, dtype=torch.bfloat16, device=gpu), normed, 1e-5, n)
  assert torch.equal(h2, out)


@pytest.mark.gpu
def test_combine_takes_exactly_the_rows_it_was_told_of(gpu):
  """Rows beyond splits x tokens x (choices + shared experts) are refused, not taken for shared experts: two K slices given as
  one, a shared expert that was not announced, and the other way round."""
  from xotorch_support_jetson_amd.ops._ext import require
  C, T, k, D = require(), 3, 2, 64
  slot_of, topw = torch.arange(T * k, dtype=torch.int32, device=gpu), torch.ones(T, k, device=gpu)
  h, lnw = torch.zeros(T, D, dtype=torch.bfloat16, device=gpu), torch.ones(D, dtype=torch.bfloat16, device=gpu)
  for rows, splits, shared, ok in ((T * k, 1, 0, True), (2 * T * k, 2, 0, True), (2 * T * (k + 1), 2, 1, True), (2 * T * k, 1, 0, False),
                                   (T * (k + 1), 1, 0, False), (T * k, 1, 1, False), (T * k, 1, -1, False), (2 * T * k, 1, 1, False)):
    y = torch.zeros(rows, D, device=gpu)
    for call in (lambda: C.moe_combine(y, slot_of, topw, h, splits, shared),
                 lambda: C.moe_combine_norm(y, slot_of, topw, h, splits, lnw, torch.empty_like(h), 1e-5, shared)):
      if ok:
        call()
      else:
        with pytest.raises(RuntimeError):
          call()


@pytest.mark.gpu
@pytest.mark.parametrize("E", [17, 64, 65, 130])
@pytest.mark.parametrize("S", [1, 2])
def test_blocks_of_64_rows_exact(gpu, E, S):
  """Experts with more than 64 rows, whose further rows are blocks of other workgroups: row counts around multiples of 64 in
  every place of a wave's search through the offsets, bit for bit on integers; no other row is written."""
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(E + S)
  cnt = torch.tensor([0, 63, 64, 65, 0, 127, 128, 129, 1, 192, 193])[torch.randint(0, 11, (E,), generator=g)]
  cnt[0], cnt[-1] = 129, 193
  off = torch.cat([torch.zeros(1, dtype=torch.long), cnt.cumsum(0)]).int()
  slots, T, N, Kd = int(off[-1]), 200, 128, 256
  x, w, tok = integers(g, T, Kd), integers(g, E, N, Kd), torch.randint(0, T, (slots,), generator=g).int()
  y = torch.full((S * slots, N), 7.0, device=gpu)
  require().gemm_moe(x.to(gpu), torch.stack([shuffle_for_stream(m.to(gpu)) for m in w]), y, off.to(gpu), tok.to(gpu), K.EPI["none"], T, True, S, 0)
  want = torch.cat([x[tok[off[e]:off[e + 1]].long()].float() @ w[e].float().t() for e in range(E)])
  assert torch.equal(y.view(S, slots, N).sum(0).cpu(), want)


@pytest.mark.gpu
def test_one_set_of_experts_is_not_slower_than_all(gpu):
  """340 tokens that all choose the same six of 64 experts read a tenth of the weights that evenly spread ones read: their rows
  side by side take less time too (82 of 131 us; 184 of 138 where one workgroup took an expert's rows one block after the other)."""
  from xotorch_support_jetson_amd.ops._ext import require
  E, k, T, N, Kd = 64, 6, 340, 2816, 2048
  x, w = torch.zeros(T, Kd, dtype=torch.bfloat16, device=gpu), torch.zeros(4, E, N, Kd, dtype=torch.bfloat16, device=gpu)
  y, took = torch.empty(T * k, N // 2, dtype=torch.bfloat16, device=gpu), []
  for cnt in ([T] * k + [0] * (E - k), [32] * 56 + [31] * 8):
    off = torch.tensor([0] + cnt).cumsum(0).int().to(gpu)
    tok = (torch.arange(T * k, device=gpu) % T).int()
    times = []
    for i in range(16):
      a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
      a.record()
      require().gemm_moe(x, w[i % 4], y, off, tok, K.EPI["silu"], T, True, 1, 0)
      b.record()
      b.synchronize()
      times.append(a.elapsed_time(b))
    took.append(sorted(times)[8])
  assert took[0] < took[1], took
