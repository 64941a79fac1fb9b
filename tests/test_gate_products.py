"""Gates of the channel-decay delta rule out of low ranks: the products on the fp32 matrix unit (ranks of whole eights) and beside it,
over token counts at the edges of a workgroup's rows, ranks that end inside a block of 32, slabs, both weight types."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R

# ranks of whole eights and others: inside a block of 32, across the four blocks that are asked for first and past them
RANKS = [(128, 128), (8, 40), (136, 16), (12, 128), (1024, 1000), (3, 5), (100, 31), (129, 255)]


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 7, 8, 9, 16, 17, 48])
@pytest.mark.parametrize("ra,rg", RANKS)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S", [1, 3, 9])
def test_gates(T, ra, rg, dt, S):
  g = torch.Generator(device="cuda").manual_seed(T + ra + rg)
  H, d, ng = 3, 40, 200

  def rnd(*s):
    return torch.randn(*s, generator=g, device="cuda")
  n = H + ra + rg + 5
  P = rnd(S, T, n) * S ** -0.5
  a2, g2 = (rnd(r, k).mul(k ** -0.5).to(dt) for r, k in ((H * d, ra), (ng, rg)))
  bias, A = rnd(H * d), rnd(H) * 0.4
  outs = [[torch.full(s, float("nan"), device=dev) for s in ((T, H), (T, H * d), (T, ng))] for dev in ("cuda", "cpu")]
  K.recurrence_gates(P if S > 1 else P[0], 0, outs[0][0], H, a2, bias, A, outs[0][1], H + ra, g2, outs[0][2])
  full = P.double().sum(0).float().cpu()
  R.recurrence_gates(full, 0, outs[1][0], H, a2.cpu(), bias.cpu(), A.cpu(), outs[1][1], H + ra, g2.cpu(), outs[1][2], None)
  for got, want in zip(*outs):
    # fp32 sums of at most 1024 terms of about rank ** -0.5 in another order: 2^-24 of partial sums of a few units each
    assert float((got.cpu() - want).abs().max()) < 2e-5
  bad = P.clone()
  bad[:, 0, H:] = float("inf")  # a row that is no number leaves the others alone
  again = [torch.empty_like(t) for t in outs[0]]
  K.recurrence_gates(bad if S > 1 else bad[0], 0, again[0], H, a2, bias, A, again[1], H + ra, g2, again[2])
  assert all(torch.equal(a[1:], b[1:]) for a, b in zip(again, outs[0]))
