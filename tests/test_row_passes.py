"""The norm passes between projections (sandwich_add_norm, resid_scale_norm, pair_norm_mean) against float64: few rows and many,
rows of one and two groups a thread, one slab to more than are asked for at once."""
import pytest
import torch


def _rms(x, eps):
  return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 64, 65])
@pytest.mark.parametrize("D", [2048, 2052, 4096, 1000])
@pytest.mark.parametrize("S", [1, 2, 12, 13, 17])
def test_against_float64(gpu, T, D, S):
  from xotorch_support_jetson_amd.ops import kernels as K
  g = torch.Generator(device=gpu).manual_seed(T + D + S)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  eps, y, y2 = 1e-5, rn(S, T, D), rn(max(1, S - 1), T, D)
  # fp32 sums of S slabs and of D squares, bf16 results: 2^-8 of the value, and of rows of unit size
  close = lambda a, b: torch.testing.assert_close(a.double(), b, rtol=8e-3, atol=1e-4)  # noqa: E731
  fine = lambda a, b: torch.testing.assert_close(a.double(), b, rtol=1e-5, atol=2e-5)  # noqa: E731
  slabs = lambda t: t[0].contiguous() if t.shape[0] == 1 else t  # noqa: E731
  x, wb, wn = rn(T, D), rn(D), rn(D)
  want = x.double() + 0.5 * _rms(y.double().sum(0), eps) * wb.double()
  h, out = x.clone(), torch.zeros(T, D + 4, dtype=torch.bfloat16, device=gpu)
  K.sandwich_add_norm(h, slabs(y), wb, wn, eps, out, mult=0.5)
  fine(h, want)
  close(out[:, :D], _rms(want, eps) * wn.double())
  assert not out[:, D:].any()

  s1, s2, gain = rn(D), rn(D), torch.full((1,), 0.7, device=gpu)
  want = x.double() + s1.double() * y.double().sum(0) + s2.double() * y2.double().sum(0)
  h, out = x.clone(), torch.zeros(T, D + 4, dtype=torch.bfloat16, device=gpu)
  K.resid_scale_norm(h, slabs(y), s1, slabs(y2), s2, gain=gain, eps=eps, out=out)
  fine(h, want)
  close(out[:, :D], _rms(want, eps) * 0.7)
  assert not out[:, D:].any()
  h = x.clone()
  K.resid_scale_norm(h, slabs(y), s1)  # one branch, no norm behind it
  fine(h, x.double() + s1.double() * y.double().sum(0))

  a, w2, mean = rn(T, D), rn(2, D), torch.empty(T, D, device=gpu)
  K.pair_norm_mean(a, slabs(y), w2, eps, mean)
  fine(mean, 0.5 * (_rms(a.double(), eps) * w2[0].double() + _rms(y.double().sum(0), eps) * w2[1].double()))
