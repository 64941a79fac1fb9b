"""The per-head gated norms of prompts (csrc/mixer_util.h gated_norm_half_k): heads that leave lanes or half waves idle, an odd token
count, rows of wider buffers, and the sizes that stay with the other kernels, against float64."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,dv", [(2048, 8, 128), (2049, 9, 128), (4097, 9, 68), (257, 3, 100), (300, 2, 64), (300, 2, 132), (255, 8, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_against_float64(gpu, T, H, dv, dtype):
  """fp32 sums of at most 132 squares (128 * 2^-24), exponentials of a few 2^-24; bf16 results one rounding (2^-9, doubled)."""
  g = torch.Generator().manual_seed(T + dv)
  o, P, w = torch.randn(T, H, dv, generator=g), torch.randn(T, H * dv + 12, generator=g), torch.randn(H * dv, generator=g)
  gate = P[:, 4:4 + H * dv].double().reshape(T, H, dv)
  unit = o.double() / torch.sqrt(o.double().square().mean(-1, keepdim=True) + 1e-5)
  rtol = 2 ** -8 if dtype == torch.bfloat16 else 2e-5
  out = torch.zeros(T, H * dv + 8, dtype=dtype, device=gpu)
  K.gated_rmsnorm(o.reshape(T, -1).to(gpu), w[:dv].to(gpu), P.to(gpu), 4, 1e-5, 0.7, out[:, :H * dv])
  want = (unit * w[:dv].double() * torch.nn.functional.silu(gate) * 0.7).reshape(T, -1)
  torch.testing.assert_close(out[:, :H * dv].cpu().double(), want, rtol=rtol, atol=1e-5)
  assert not out[:, H * dv:].any()
  K.gated_group_norm(o.reshape(T, -1).to(gpu), None, w.to(gpu), P.to(gpu), 4, H, 1e-5, out)
  want = (unit * w.double().reshape(H, dv) * torch.sigmoid(gate)).reshape(T, -1)
  torch.testing.assert_close(out[:, :H * dv].cpu().double(), want, rtol=rtol, atol=1e-5)
