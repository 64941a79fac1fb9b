"""Latent attention's norm, rotation and cache write on split-K slabs, against the slab sum followed by the kernel of longer steps."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops.rope import build_cos_sin


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 37, 128])
@pytest.mark.parametrize("S", [1, 3, 4, 9])
@pytest.mark.parametrize("H,dn,DL,DR,pad", [(16, 128, 512, 64, 0), (3, 72, 256, 16, 40), (40, 128, 512, 64, 64), (1, 8, 2048, 32, 8)])
def test_slabs_against_the_reduced_rows(T, S, H, dn, DL, DR, pad):
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator(device="cuda").manual_seed(T + S)
  nope, nq = H * dn, H * (dn + DR)
  N = nq + DL + DR + pad
  P = torch.randn(S, T, N, generator=g, device="cuda")
  ln = torch.randn(DL, generator=g, device="cuda").bfloat16()
  pos = torch.randint(-1, 70, (T,), generator=g, device="cuda").int()  # (clamped to the table)
  slots = torch.randperm(3 * 64, generator=g, device="cuda")[:T]
  slots[T // 2] = -1 if T > 1 else 5
  if T > 2:
    slots[1] = 3 * 64  # beyond the cache
  tab = build_cos_sin(DR, 64, 10000.0, None, device="cuda")
  total = P[0].clone()
  for s in range(1, S):
    total += P[s]
  A = total.bfloat16()
  want_c, got_c = (torch.zeros(3, 64, DL + DR, dtype=torch.bfloat16, device="cuda") for _ in range(2))
  q = torch.full((T, nq + 8), 3.0, dtype=torch.bfloat16, device="cuda")
  require().mla_prep_slabs(P if S > 1 else P[0], nope, ln, q, H, pos, tab, slots, got_c, 1e-6)
  K.mla_prep(A[:, nq:], ln, A, nope, H, pos, tab, slots, want_c, 1e-6)
  assert torch.equal(q[:, :nope], A[:, :nope]) and bool((q[:, nq:] == 3.0).all())
  # (rotations: products contracted differently, at most the last bf16 place of a pair's scale)
  torch.testing.assert_close(q[:, nope:nq], A[:, nope:nq], rtol=8e-3, atol=2e-2)
  torch.testing.assert_close(got_c, want_c, rtol=8e-3, atol=2e-2)
  assert torch.equal(got_c.abs().sum(-1) > 0, want_c.abs().sum(-1) > 0)
