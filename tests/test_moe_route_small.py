"""Expert routing of few tokens in one launch against the general kernels, which take over above 128 tokens: the same choices and
weights bit for bit, also for ties, infinities and rows that are not numbers; and the router's product over split experts."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K


def rows(T, E, seed):
  lg = torch.randn(T, E, generator=torch.Generator().manual_seed(seed)) * 3
  lg[::5] = lg[::5].round()  # ties
  if T > 3:
    lg[1, : E // 2] = float("-inf")
    lg[2] = float("nan")
    lg[3, 0], lg[3, -1] = float("inf"), float("nan")
  return lg.cuda()


def check_slots(topi, slot_of, sorted_tok, off, T, k, E):
  topi, slot_of, sorted_tok, off = (t.cpu().long() for t in (topi, slot_of, sorted_tok, off))
  assert torch.equal(off[:E + 1], torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(topi, minlength=E).cumsum(0)]))
  assert torch.equal(slot_of.sort().values, torch.arange(T * k))
  assert torch.equal(sorted_tok[slot_of], torch.arange(T * k) // k)
  assert bool(((slot_of >= off[topi]) & (slot_of < off[topi + 1])).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 15, 16, 17, 37, 128])
@pytest.mark.parametrize("E,k,sig,norm,bias", [(64, 6, False, False, False), (64, 16, True, True, True), (4, 4, False, True, False),
                                               (33, 1, True, False, True), (1, 1, False, False, False), (63, 8, False, False, True)])
def test_scores_and_bias(T, E, k, sig, norm, bias):
  lg = rows(T, E, T + E)
  b = torch.linspace(-0.2, 0.2, E).cuda() if bias else None
  big = torch.cat([lg, rows(129, E, 7)])
  few = K.moe_route_ds(lg, b, k, 1, 1, 0, sig, norm, 1.5)
  many = K.moe_route_ds(big, b, k, 1, 1, 0, sig, norm, 1.5)
  assert torch.equal(few[1], many[1][:T * k])
  assert torch.equal(few[0].view(torch.int32), many[0][:T * k].view(torch.int32)) or torch.equal(
    few[0].nan_to_num(nan=123.0), many[0][:T * k].nan_to_num(nan=123.0))
  check_slots(few[1], *few[2:], T, k, E)
  check_slots(many[1], *many[2:], T + 129, k, E)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 16, 17, 37, 300, 2100])
@pytest.mark.parametrize("E,D", [(32, 512), (64, 2048), (64, 1536), (128, 1024), (160, 5120), (256, 7168), (256, 512)])
def test_router_product(T, E, D):
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(E + T)
  x, w = torch.randint(-2, 3, (T, D), generator=g).bfloat16().cuda(), torch.randint(-2, 3, (E, D), generator=g).bfloat16().cuda()
  out = torch.empty(T, E, device="cuda")
  require().router_logits(x, w, out)
  assert torch.equal(out, x.float() @ w.float().t())  # (integers below 2^24: exact in every order)
