"""Decode attention of models with routed experts: pages summed one behind the other, partitions merged in order, whatever the
batch, so that an almost tied token keeps its experts."""
import math

import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R


def wave_pages(batch, hkv, pages):
  n = max(1, min(max(pages // 2, 1), -(-1024 // (batch * hkv))))
  return -(-pages // max(n, -(-pages // 32)))


def test_routed_partitions():
  for W in (1, 9, 33, 64, 130):
    ws = K.DecodeWorkspace(200, 32, 128, W * 64, torch.device("meta"), algo=-1, routed=True)
    for b in (1, 2, 7, 8, 9, 24, 64, 128, 200):
      for hkv in (1, 2, 8):
        ppp, nparts, algo = ws.partition(b, hkv, W)
        big = b * hkv * W * 64 * 128 * 4 >= K.NT_MIN_KV_BYTES
        assert algo == (0 if b * hkv < 64 else 8 if big else 7)
        assert ppp * nparts >= W > ppp * (nparts - 1)
        assert algo == 0 or ppp == wave_pages(b, hkv, W)
  plain = K.DecodeWorkspace(64, 32, 128, 512, torch.device("meta"), algo=-1)
  assert plain.partition(64, 8, 8)[2] == 2


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hkv,Dh", [(32, 8, 128), (16, 8, 64), (16, 1, 128)])
@pytest.mark.parametrize("width", [1, 8, 21, 40])
def test_routed_order(H, Hkv, Dh, width):
  """Against float32, and bit for bit the order of the lone wave without a prefetch (algo 1) over the same partitions."""
  g = torch.Generator(device="cuda").manual_seed(width)
  full = width * 64
  lens = sorted({1, 63, 64, 65, 129, 300, full - 1, full} & set(range(1, full + 1)))
  lens = (lens * 9 + [0]) if Hkv > 1 else lens * 20
  B, pages = len(lens), sum(-(-n // 64) for n in lens) + 1
  kc = torch.randn(pages, Hkv, 64, Dh, generator=g, device="cuda").bfloat16()
  vc = torch.randn(pages, Hkv, Dh, 64, generator=g, device="cuda").bfloat16()
  bt, at = torch.zeros(B, width, dtype=torch.int32), 0
  perm = torch.randperm(pages, generator=g, device="cuda").int().cpu()
  for i, n in enumerate(lens):
    m = -(-n // 64)
    bt[i, :m] = perm[at:at + m]
    at += m
  bt, cl = bt.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda")
  q = torch.randn(B, H, Dh, generator=g, device="cuda").bfloat16()
  ws = K.DecodeWorkspace(B, H, Dh, full, q.device, algo=-1, routed=True)
  ppp, _, algo = ws.partition(B, Hkv, width)
  out = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws)
  live = [i for i, n in enumerate(lens) if n]
  want = R.attn_decode(q[live], kc, vc, bt[live], cl[live], 1 / math.sqrt(Dh)).float()
  # probabilities and results in bf16 (2^-9 each, of values at most a few): as for the other decode kernels
  assert float((out[live].float() - want).abs().max()) < 2e-2 * float(want.abs().max())
  assert all(float(out[i].abs().max()) == 0.0 for i, n in enumerate(lens) if not n)
  if algo:
    one = K.DecodeWorkspace(B, H, Dh, full, q.device, pages_per_part=ppp, algo=1)
    assert torch.equal(K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, one), out)


@pytest.mark.gpu
def test_models_with_routed_experts_take_it():
  from xotorch_support_jetson_amd.inference.shard import Shard
  from xotorch_support_jetson_amd.models.config import preset
  from xotorch_support_jetson_amd.runtime.runner import ShardRunner
  for name, routed in (("tiny-mixtral", True), ("tiny-llama", False)):
    c = preset(name)
    r = ShardRunner(c, Shard(name, 0, c.num_layers - 1, c.num_layers), "cuda:0", num_pages=8, max_batch=2, max_ctx=128)
    assert r.model.ws.routed is routed
