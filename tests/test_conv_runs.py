"""Convolutions over runs of tokens: SiLU and the norms of eight tokens at a time against float64, at heads of every width and ragged runs."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R


@pytest.mark.gpu
@pytest.mark.parametrize("head", [7, 64, 100, 128, 200, 256])
@pytest.mark.parametrize("lens", [[3, 1, 8], [9, 40, 17], [1100]])
def test_units(head, lens):
  parts = [(head, R.CONV_SILU | R.CONV_UNIT_SCALED), (head, R.CONV_SILU | R.CONV_UNIT), (head, R.CONV_UNIT), (head, R.CONV_SILU)]
  C, T, B = 4 * head, sum(lens), len(lens)
  units, width = R.conv_units(parts, C)
  g = torch.Generator().manual_seed(head + T)
  P, w, state = 4 * torch.randn(T, C, generator=g), torch.randn(C, 4, generator=g), torch.randn(B, 3, C, generator=g)
  P[::5] *= 30  # (SiLU's ends: e^-x past every float, and nothing)
  cu = torch.tensor([0] + lens).cumsum(0).int()
  out, S = torch.full((T, C), float("nan"), device="cuda"), state.cuda()
  K.conv_prep(P.cuda(), 0, w.cuda(), None, units.cuda(), None, S, torch.arange(B, dtype=torch.int32, device="cuda"), cu.cuda(), 1e-5, out, max(lens), width)
  for b, n in enumerate(lens):
    x = torch.cat([state[b], P[cu[b]:cu[b + 1]]]).double()
    y = sum(w[:, j].double() * x[j:j + n] for j in range(4))
    size = sum(w[:, j].double().abs() * x[j:j + n].abs() for j in range(4))  # four products and sums, then SiLU with a slope up to 1.1
    for i, (_, kind) in enumerate(parts):
      at = slice(i * head, (i + 1) * head)
      u = torch.nn.functional.silu(y[:, at]) if kind & R.CONV_SILU else y[:, at]
      err = 2**-24 * (6 * size[:, at] + 8 * u.abs())
      if kind & ~R.CONV_SILU:
        f = 1 / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6) * (head**-0.5 if kind & R.CONV_UNIT_SCALED else 1)
        err = f * (err + u.abs() * f * (err.norm(dim=-1, keepdim=True) if not kind & R.CONV_UNIT_SCALED else err.norm(dim=-1, keepdim=True) * head**0.5)) + 2**-20 * (u * f).abs()
        u = u * f
      assert ((out[cu[b]:cu[b + 1], at].cpu().double() - u).abs() <= err + 1e-30).all(), (b, i)
