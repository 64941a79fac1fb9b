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


@pytest.mark.gpu
@pytest.mark.parametrize("head", [1, 7, 64, 66, 126, 128, 130, 256])
@pytest.mark.parametrize("off", [0, 1, 2])
@pytest.mark.parametrize("taps,lens", [(4, [5, 1, 37]), (2, [1030, 0, 9]), (1, [33]), (6, [70, 3])])  # (runs or units as neighbours)
def test_whole_rows_as_two_slabs(head, off, taps, lens):
  """Rows loaded without a branch (whole vectors, unsplit) and any others: the same numbers as the sum of the rows and of nothing."""
  C, T, B = 3 * head, sum(lens), len(lens)
  units, width = R.conv_units([(head, R.CONV_SILU | R.CONV_UNIT), (head, R.CONV_SILU), (head, 0)], C)
  g = torch.Generator(device="cuda").manual_seed(head + off)
  rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
  P, w, state = rn(T, C + 4), rn(C, taps), rn(B, taps - 1, C)
  cu, slots, got = torch.tensor([0] + lens).cumsum(0).int().cuda(), torch.arange(B, dtype=torch.int32, device="cuda"), []
  for rows in (P, torch.stack([P, torch.zeros_like(P)])):
    S, out = state.clone(), torch.full((T, C), float("nan"), device="cuda")
    K.conv_prep(rows, off, w, None, units.cuda(), None, S, slots, cu, 1e-5, out, max(lens), width)
    got.append((out, S))
  assert all(torch.equal(a, b) for a, b in zip(*got)) and not got[0][0].isnan().any()


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [True, False])
def test_silu_of_any_input(runs):
  """SiLU where e^-x leaves the range of a float: -0 or 0 for finite inputs, however large, and infinities and no numbers as a
  quotient has them."""
  inf, nan = float("inf"), float("nan")
  v = [-inf, -3e38, -1e35, -1e30, -1e4, -129.0, -128.0, -100.0, -89.0, -88.0, -87.5, -87.0, -80.0, -1.0, -1e-30, 0.0, 1e-30, 1.0, 80.0, 87.0, 100.0, 1e35, 3e38, inf, nan]
  x = torch.tensor([v, v[::-1], v], dtype=torch.float32, device="cuda")
  T, C = x.shape
  units, width = R.conv_units([(C, R.CONV_SILU)], C)
  out, slots = torch.zeros_like(x), torch.arange(1 if runs else T, dtype=torch.int32, device="cuda")
  cu = torch.tensor([0, T] if runs else list(range(T + 1)), dtype=torch.int32, device="cuda")
  K.conv_prep(x, 0, torch.ones(C, 1, device="cuda"), None, units.cuda(), None, torch.zeros(len(slots), 0, C, device="cuda"), slots, cu, 1e-5, out,
              T if runs else 1, width)
  got, x = out.double().cpu(), x.double().cpu()
  want = x / (1 + torch.exp(-x))
  want[(x < -700) & (x > -inf)] = 0.0  # (e^-x past float64)
  assert torch.equal(got.isnan(), want.isnan())
  ok = ~want.isnan()
  got, want, x = got[ok], want[ok], x[ok]
  assert torch.equal(got.isinf(), want.isinf()) and bool((got[got.isinf()] > 0).all())
  fin = ~want.isinf()
  got, want, x = got[fin], want[fin], x[fin]
  # 2^-22 of the value (twice the 1.7e-7 of ordinary ones); between -88.8 and -87.3 the reciprocal may be 0, below it is
  assert bool(((got - want).abs() <= 2.0 ** -22 * want.abs() + torch.where(x < -87.3, 1.2e-36, 0.0)).all())
  assert bool((got[x < -88.8] == 0).all())
