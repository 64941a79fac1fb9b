"""Decode attention by the waves of a workgroup together (algo 2 / 3): edges of pages, waves without a page, empty contexts,
partitions, one and four waves, every group size."""
import math

import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R


def test_workspace_holds_every_partitioning():
  for W in (1, 9, 17, 33, 64, 65, 130):
    ws = K.DecodeWorkspace(40, 32, 128, W * 64, torch.device("meta"), algo=-1)
    for b in range(1, 41):
      for hkv in (1, 2, 4, 8, 16):
        for w in {x for x in (8, 16, 32) if x < W} | {W}:
          ppp, nparts, _ = ws.partition(b, hkv, w)
          assert ppp * nparts >= w > ppp * (nparts - 1)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hkv,Dh", [(8, 8, 64), (32, 8, 128), (16, 1, 128), (14, 2, 64)])
@pytest.mark.parametrize("width,ppp", [(8, None), (8, 3), (21, None), (21, 21), (70, None)])
def test_group_kernel(H, Hkv, Dh, width, ppp):
  g = torch.Generator(device="cuda").manual_seed(H + width)
  full = width * 64
  ctx = sorted({1, 63, 64, 65, 128, 129, 255, 257, 511, min(full, 1300), full - 1, full} & set(range(1, full + 1))) + [0]
  # a step that fills the chip with units (one wave each over short tables), and one that does not
  for rep in (1, 1 + 1024 // (Hkv * len(ctx))) if width == 8 and ppp is None else (1,):
    lens = ctx * rep
    B = len(lens)
    pages = sum(-(-n // 64) for n in ctx) + 1
    kc = torch.randn(pages, Hkv, 64, Dh, generator=g, device="cuda").bfloat16()
    vc = torch.randn(pages, Hkv, Dh, 64, generator=g, device="cuda").bfloat16()
    perm, at = torch.randperm(pages, generator=g, device="cuda").int(), 0
    bt = torch.zeros(len(ctx), width, dtype=torch.int32, device="cuda")
    for i, n in enumerate(ctx):
      m = -(-n // 64)
      bt[i, :m] = perm[at:at + m]
      at += m
    bt, cl = bt.repeat(rep, 1).contiguous(), torch.tensor(lens, dtype=torch.int32, device="cuda")
    q = torch.randn(B, H, Dh, generator=g, device="cuda").bfloat16()
    n1 = len(ctx) - 1  # (the empty context's row is zeros)
    want = R.attn_decode(q[:n1], kc, vc, bt[:n1], cl[:n1], 1 / math.sqrt(Dh)).float()
    for algo in (2, 3):
      ws = K.DecodeWorkspace(B, H, Dh, full, q.device, pages_per_part=ppp, algo=algo)
      out = K.attn_decode(q, kc, vc, bt, cl, 1 / math.sqrt(Dh), ws).float()
      # probabilities and results in bf16 (2^-9 each, of values at most a few): as for the other decode kernels
      assert float((out[:n1] - want).abs().max()) < 2e-2 * float(want.abs().max()), (algo, rep)
      assert float(out[n1].abs().max()) == 0.0 and bool(torch.isfinite(out).all())
      assert torch.equal(K.attn_decode(q, kc, vc, bt, cl, 1 / math.sqrt(Dh), ws).float(), out)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hkv,Dh", [(32, 8, 64), (64, 8, 128), (16, 1, 128)])
@pytest.mark.parametrize("width", [1, 3, 8])
def test_short_tables_of_large_batches_take_one_wave_a_unit(H, Hkv, Dh, width):
  """1024 and more units over at most 8 pages: bit for bit the lone wave without a prefetch (algo 1)."""
  g = torch.Generator(device="cuda").manual_seed(width)
  B = 1024 // Hkv
  cl = torch.randint(0, width * 64 + 1, (B,), generator=g, device="cuda", dtype=torch.int32)
  pages = 40
  kc = torch.randn(pages, Hkv, 64, Dh, generator=g, device="cuda").bfloat16()
  vc = torch.randn(pages, Hkv, Dh, 64, generator=g, device="cuda").bfloat16()
  bt = torch.randint(0, pages, (B, width), generator=g, device="cuda", dtype=torch.int32)
  q = torch.randn(B, H, Dh, generator=g, device="cuda").bfloat16()
  one = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, K.DecodeWorkspace(B, H, Dh, width * 64, q.device, pages_per_part=width, algo=1))
  for algo in (2, 3):
    ws = K.DecodeWorkspace(B, H, Dh, width * 64, q.device, algo=algo)
    assert ws.partition(B, Hkv, width)[1] == 1
    assert torch.equal(K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws), one)


def test_partitions_leave_at_most_one_unit_a_cu():
  """Contexts of up to 64 pages are cut only while (sequence, KV head, partition) units do not outnumber the 256 CUs."""
  for batch in range(1, 128):
    for hkv in (1, 2, 3, 8, 16):
      for pages in (1, 8, 9, 16, 32, 64):
        parts = K.group_parts(batch, hkv, pages)
        assert parts == 1 or batch * hkv * parts <= 256
        assert parts <= -(-pages // 4)
