"""K slices of the weight-streaming GEMM that are no power of two: exact integer sums through every reader of the slabs."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L


def test_offered_splits():
  for M in (1, 2, 48):
    for k in (128, 384, 1408, 2816, 5632, 4096, 13824):
      got = {S for ntw, S in L.GemmPolicy._stream_cands(M, 256, k, "none") if ntw == 1}
      assert 1 in got and all(k % (128 * S) == 0 for S in got) and max(got) <= (16 if M > 1 else 8)
      assert {S for S in (1, 2, 4, 8) if k % (128 * S) == 0} <= got
  assert 11 in {S for _, S in L.GemmPolicy._stream_cands(48, 2048, 5632, "none")}


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 17, 48])
@pytest.mark.parametrize("S", [3, 5, 7, 9, 11, 16])
def test_slabs_add_up(M, S):
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(S)
  N, Kd = 256, 256 * S
  x = torch.randint(-2, 3, (M, Kd), generator=g).bfloat16().cuda()
  w = torch.randint(-1, 2, (N, Kd), generator=g).bfloat16().cuda()
  want = x.float() @ w.float().t()  # (integers below 2^24: every order of the sum is exact)
  ws = L.to_stream_layout(w)
  for ntw in (1, 2):
    y = torch.empty(M, N, device="cuda")
    L._shuffled_call(x, ws, None, None, "none", y, ("stream", ntw, S))
    assert torch.equal(y, want)
    slabs = L.scratch.splitk(x.device, S * M * N)
    require().gemm_stream(x, ws, y, None, None, slabs, K.EPI["none"], ntw, S, True, False)
    assert torch.equal(slabs[:S * M * N].view(S, M, N).sum(0), want)
    # the residual norm that sums the slabs, against the product rounded in one piece
    h = torch.randint(-8, 9, (M, N), generator=g).bfloat16().cuda()
    lnw, out, h2 = torch.ones(N, device="cuda").bfloat16(), torch.empty(M, N, device="cuda").bfloat16(), h.clone()
    require().splitk_resid_rmsnorm(slabs, S, None, h2, lnw, out, 1e-5)
    assert torch.equal(h2, (want + h.float()).bfloat16())
  act = torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda")
  L._shuffled_call(x, ws, None, None, "silu", act, ("stream", 2, S))
  t = want.view(M, N // 32, 2, 16)
  ref = (torch.nn.functional.silu(t[:, :, 0].double()) * t[:, :, 1].double()).reshape(M, N // 2)
  # half a bf16 step and the fp32 exponential's error
  assert bool(((act.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-5 * ref.abs().max()).all())
