"""Four-wave GEMM (csrc/gemm_w4.hip) with more than three rounds of tiles: one workgroup a CU takes tile after tile."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L
from xotorch_support_jetson_amd.ops._ext import require
from xotorch_support_jetson_amd.train import autograd_ops as A


def product(x, w, epi, dtype, bias=None, residual=None, arg=0.0):
  out = torch.empty(x.shape[0], w.shape[0] // 2 if epi in K.GLU_EPI else w.shape[0], dtype=dtype, device=x.device)
  require().gemm_big(x, w, out, bias, residual, None, K.EPI[epi], 4256, 1, True, arg)
  return out


@pytest.mark.gpu
@pytest.mark.parametrize("epi,dtype", [("none", torch.bfloat16), ("none", torch.float32), ("resid", torch.bfloat16), ("silu", torch.bfloat16),
                                       ("clamp_glu", torch.bfloat16), ("gelu_glu", torch.bfloat16), ("relu2", torch.bfloat16)])
@pytest.mark.parametrize("tall", [1535, 2561, 3073, 4000])  # ragged last row tiles; tile counts of no whole rounds
@pytest.mark.parametrize("Kd,pad", [(128, 0), (384, 24)])  # two stages a tile, and more; rows of X apart
def test_rows_of_many_tiles_as_rows_of_few(gpu, epi, dtype, tall, Kd, pad):
  """The tiles sum K in one order, so a product is bit for bit that of its rows in portions of one round, which float32 checks."""
  N, g = 96 * 256, torch.Generator(device=gpu).manual_seed(tall + Kd)
  x = torch.randn(tall, Kd + pad, device=gpu, generator=g).to(torch.bfloat16)[:, :Kd]
  w = (torch.randn(N, Kd, device=gpu, generator=g) / Kd ** 0.5).to(torch.bfloat16)
  ws = L.to_stream_layout(w)
  bias = torch.randn(N, device=gpu, generator=g).to(torch.bfloat16) if epi in ("none", "silu") else None
  res = torch.randn(tall, N, device=gpu, generator=g).to(torch.bfloat16) if epi == "resid" else None
  arg = 7.0 if epi == "clamp_glu" else 0.0
  for _ in range(2):
    out = product(x, ws, epi, dtype, bias, res, arg)
    for a in range(0, tall, 300):
      b = min(tall, a + 300)
      part = product(x[a:b], ws, epi, dtype, bias, None if res is None else res[a:b], arg)
      assert torch.equal(out[a:b], part), a
  if epi in ("none", "resid"):
    want = x[-70:].float() @ w.float().T + (bias.float() if bias is not None else res[-70:].float())
    tol = 2 ** -8 if dtype == torch.bfloat16 else 1e-5  # the result's rounding; sums of up to 384 products of size one in fp32
    torch.testing.assert_close(out[-70:].float(), want, rtol=tol, atol=1e-5 * Kd ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [64, 128, 192, 320, 2560, 2624])  # one stage a tile (a workgroup each), two, and odd numbers: the
# buffers change places; the most of tile after tile, and more
@pytest.mark.parametrize("M,N", [(8192, 6400), (7680, 6656)])  # 800 and 780 tiles
@pytest.mark.parametrize("accumulate", [False, True])
def test_weight_gradients_of_many_tiles(gpu, tokens, M, N, accumulate):
  g = torch.Generator(device=gpu).manual_seed(tokens + M)
  dy, x = (torch.randn(tokens, n, device=gpu, generator=g).to(torch.bfloat16) for n in (M, N))
  start = torch.randn(M, N, device=gpu, generator=g).to(torch.bfloat16)
  for _ in range(2):
    out = start.clone()
    assert A.dw_tn(dy, x, out, accumulate)
    for a in range(0, M, 1536):  # (fewer tiles: a workgroup each)
      b = min(M, a + 1536)
      part = start[a:b].clone()
      assert A.dw_tn(dy[:, a:b], x, part, accumulate) and torch.equal(out[a:b], part), a
  want = dy[:, -300:].float().T @ x.float() + (start[-300:].float() if accumulate else 0)
  torch.testing.assert_close(out[-300:].float(), want, rtol=2 ** -8, atol=1e-5 * tokens ** 0.5)  # (the result's rounding; fp32 sums)
