"""Values of many tokens written in whole 8-key chunks wherever they lie: sequences of any length and start behind one another, tokens
without a slot, against the token-by-token kernel of short steps."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops.rope import build_cos_sin


@pytest.mark.gpu
@pytest.mark.parametrize("Dh,Hkv", [(64, 2), (128, 1)])
@pytest.mark.parametrize("lens,starts", [([3, 70, 1, 130, 64, 9], [0, 5, 63, 8, 0, 60]), ([256], [0]), ([300], [7]), ([1] * 260, [0] * 260),
                                         ([129, 129], [1, 0])])
def test_pieces(Dh, Hkv, lens, starts):
  H = 2 * Hkv
  g = torch.Generator().manual_seed(sum(lens))
  slots, base = [], 0
  for n, s in zip(lens, starts):  # pages of a sequence in scrambled order
    pages = -(-(s + n) // 64)
    order = torch.randperm(pages, generator=g) + base
    slots += [int(order[(s + i) // 64]) * 64 + (s + i) % 64 for i in range(n)]
    base += pages
  T = len(slots)
  slots = torch.tensor(slots)
  for drop in (False, True):
    if drop:
      slots[torch.randint(0, T, (T // 7 + 1,), generator=g)] = -1
      slots[-1] = base * 64 + 5  # beyond the cache: not written
    qkv = torch.randn(T, (H + 2 * Hkv) * Dh, generator=g).bfloat16().cuda()
    pos = (torch.arange(T) % 50).int().cuda()
    tab = build_cos_sin(Dh, 64, 10000.0, None, device="cuda")
    res = []
    for step in (T, 100):  # one call; calls short enough for single tokens
      kc = torch.zeros(base, Hkv, 64, Dh, dtype=torch.bfloat16, device="cuda")
      vc = torch.zeros(base, Hkv, Dh, 64, dtype=torch.bfloat16, device="cuda")
      q = torch.cat([K.rope_kv_write(qkv[a:a + step].contiguous(), pos[a:a + step].contiguous(), tab, slots[a:a + step].cuda(), kc, vc,
                                     H, Hkv).reshape(-1, H * Dh) for a in range(0, T, step)])
      res.append((q, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*res))
