"""Grouped expert GEMMs (csrc/gemm_group.hip and the grouped order of csrc/gemm_big.hip): experts without rows, row counts at the
edges of every row tile, K slices, gathered rows, and the rule that picks a kernel."""
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
