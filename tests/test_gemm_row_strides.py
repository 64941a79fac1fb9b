"""Products of 1024 and more rows (csrc/gemm_w4.hip) whose rows of X repeat (stride 0) or overlap (stride below K)."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L
from xotorch_support_jetson_amd.ops._ext import require


def rows_of(M, Kd, ld, g, gpu):
  base = torch.randn((M - 1) * ld + Kd, device=gpu, generator=g).to(torch.bfloat16)
  return base.as_strided((M, Kd), (ld, 1))


def weights(N, Kd, g, gpu):
  w = (torch.randn(N, Kd, device=gpu, generator=g) / Kd ** 0.5).to(torch.bfloat16)
  return w, L.to_stream_layout(w)


# a result's rounding (bf16), and the sums of Kd products of size 1 / Kd ** 0.5 in fp32 (below 1e-5 of a unit)
def close(got, want):
  torch.testing.assert_close(got.float(), want, rtol=2 ** -8 if got.dtype == torch.bfloat16 else 1e-5, atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("ld", [0, 8, 256, 512, 520])  # repeated, overlapping (the last 8 and half), side by side, apart; K is 512
@pytest.mark.parametrize("M", [1100, 1024, 2561])
def test_rows_that_repeat_or_overlap(gpu, M, ld):
  g, N, Kd = torch.Generator(device=gpu).manual_seed(M + ld), 2048, 512
  x, (w, ws) = rows_of(M, Kd, ld, g, gpu), weights(N, Kd, g, gpu)
  want = x.float() @ w.float().T
  close(L.linear(x, ws), want)
  y = L.linear_slabs(x, ws)
  close(y.sum(0) if y.dim() == 3 else y, want)
  h, ln = torch.randn(M, N, device=gpu, generator=g).to(torch.bfloat16), torch.ones(N, dtype=torch.bfloat16, device=gpu)
  want = want + h.float()
  L.linear_resid_norm(x, ws, h, ln, 1e-5)
  close(h, want)


@pytest.mark.gpu
@pytest.mark.parametrize("ld", [0, 8, 128])
@pytest.mark.parametrize("tile,parts", [(4256, 1), (1280000 + 4256, 1), (1600000 + 4256, 1), (2560000 + 4256, 1), (4256, 2), (4256, 3)])
@pytest.mark.parametrize("M,N", [(300, 256), (2561, 96 * 256)])  # a few tiles; tile after tile
def test_every_row_height_and_split(gpu, ld, tile, parts, M, N):
  g, Kd = torch.Generator(device=gpu).manual_seed(M + ld), 384
  x, (w, ws) = rows_of(M, Kd, ld, g, gpu), weights(N, Kd, g, gpu)
  out = torch.empty(M, N, dtype=torch.float32, device=gpu)
  slabs = torch.empty(parts, M, N, device=gpu) if parts > 1 else None
  require().gemm_big(x, ws, out, None, None, slabs, K.EPI["none"], tile, parts, True, 0.0)
  close(out, x.float() @ w.float().T)
