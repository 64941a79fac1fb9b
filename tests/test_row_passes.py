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


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,D,Kd,parts", [(1025, 512, 512, 2048, 3), (1200, 2048, 2000, 2048, 3), (1663, 2048, 2048, 4096, 2), (1024, 4096, 4096, 2048, 2),
                                            (2049, 2048, 2048, 2048, 1)])
def test_tall_products_read_as_slabs(gpu, M, N, D, Kd, parts):
  """Products of 1024 and more rows left in parts of K (linear_slabs, linear_resid_norm), ragged last row tiles, two branches in the two
  slots: every pass that sums them against float64."""
  from xotorch_support_jetson_amd.ops import kernels as K
  from xotorch_support_jetson_amd.ops import linear as L
  g = torch.Generator(device=gpu).manual_seed(M + N)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  eps, k2 = 1e-5, 2048
  x, x2 = rn(M, Kd).bfloat16(), rn(M, k2).bfloat16()
  w, w2 = (rn(N, Kd) / Kd ** 0.5).bfloat16(), (rn(N, k2) / k2 ** 0.5).bfloat16()
  ws, ws2 = L.to_stream_layout(w), L.to_stream_layout(w2)
  y, y2 = x.double() @ w.double().T, x2.double() @ w2.double().T
  slabs = lambda: L.linear_slabs(x, ws)  # noqa: E731
  # fp32 sums of Kd products of size Kd^-1/2: 6e-8 Kd^1/2 = 4e-6 rms, the largest of 3e6 values 5.5 times that, before unit-size norms;
  # bf16 results: 2^-8 of the value
  fine = lambda a, b: torch.testing.assert_close(a.double(), b, rtol=1e-5, atol=4e-5)  # noqa: E731
  close = lambda a, b: torch.testing.assert_close(a.double(), b, rtol=8e-3, atol=1e-4)  # noqa: E731

  h0, s1, s2, gain, wb, wn = rn(M, D), rn(D), rn(D), torch.full((1,), 0.7, device=gpu), rn(D), rn(D)
  b = L.linear_slabs(x2, ws2, slot=1)
  a = slabs()
  assert (a.shape, b.dim()) == ((parts, M, N) if parts > 1 else (M, N), 3 if parts > 1 else 2)
  h, out = h0.clone(), torch.empty(M, D, dtype=torch.bfloat16, device=gpu)
  K.resid_scale_norm(h, a, s1, b, s2, gain=gain, eps=eps, out=out)
  want = h0.double() + s1.double() * y[:, :D] + s2.double() * y2[:, :D]
  fine(h, want)
  close(out, _rms(want, eps) * 0.7)

  h = h0.clone()
  K.sandwich_add_norm(h, slabs(), wb, wn, eps, out)
  want = h0.double() + _rms(y[:, :D], eps) * wb.double()
  fine(h, want)
  close(out, _rms(want, eps) * wn.double())

  mean, both = torch.empty(M, D, device=gpu), rn(2, D)
  K.pair_norm_mean(h0, slabs(), both, eps, mean)
  fine(mean, 0.5 * (_rms(h0.double(), eps) * both[0].double() + _rms(y[:, :D], eps) * both[1].double()))

  e, slot, top = rn(M, D), torch.randperm(M, generator=g, device=gpu).int(), rn(M, 1)
  K.moe_weighted_sum(e, slot, top, 1, slabs(), None, 0, mean)
  fine(mean, e.double()[slot.long()] * top.double() + y[:, :D])

  table, ids = rn(9, 256).bfloat16(), torch.arange(M, device=gpu).int() % 9
  act = torch.empty(M, 256, dtype=torch.bfloat16, device=gpu)
  K.gelu_gather_mul(slabs(), 100, table, ids, 3, 250, act)
  close(act[:, :250], torch.nn.functional.gelu(y[:, 100:350], approximate="tanh") * table[ids.long(), 3:253].double())

  hb, ln, bias = rn(M, N).bfloat16(), rn(N).bfloat16(), rn(N).bfloat16()
  want = hb.double() + y + bias.double()
  out = L.linear_resid_norm(x, ws, hb, ln, eps, bias=bias)
  close(hb, want)
  torch.testing.assert_close(out.double(), _rms(want, eps) * ln.double(), rtol=2e-2, atol=1e-3)  # (of the rounded row, rounded again)
