"""Steps of single tokens through a recurrence and the per-head norm behind it (recurrence_norm): the one-launch form
(csrc/recurrence_step.hip) and the sizes it leaves to the general kernels, against the plain fp32 form."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K


def inputs(mode, B, H, G, d, dv, seed):
  """Arguments of recurrence_norm on the CPU; q | k | v are slices of wider rows, one sequence has no slot."""
  g = torch.Generator().manual_seed(seed)
  rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
  P = rn(B, 2 * G * d + 2 * H * dv + 24)
  q, k, v, gate = P.split([G * d, G * d, H * dv, H * dv + 24], 1)  # (a gate's rows may be wider)
  k = torch.nn.functional.normalize(k.reshape(B, G, d), dim=-1).reshape(B, G * d)
  slots = torch.randperm(B + 2, generator=g)[:B].int()
  if B > 2:
    slots[1] = -1
  beta = torch.sigmoid(rn(B, H)) if mode != "gla" else None
  decay = {"delta": lambda: torch.sigmoid(rn(B, H) + 2), "channel": lambda: torch.sigmoid(rn(B, H * d) + 2), "gla": lambda: None}[mode]()
  gla = (P, P.shape[1] - 24, rn(H * d, 20) * 0.2, rn(H * d) + 2, 16.0) if mode == "gla" else None
  w = rn(H * dv if mode == "channel" else dv)
  return dict(q=q, k=k, v=v, decay=decay, beta=beta, q_scale=d ** -0.5, state=rn(B + 2, H, dv, d), state_slots=slots,
              cu_q=torch.arange(B + 1, dtype=torch.int32), w=w, gate=gate, sigmoid=mode == "channel", eps=1e-5,
              scale=1.0 if mode == "channel" else 0.7, gla=gla, max_qlen=1)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["delta", "channel", "gla"])
@pytest.mark.parametrize("H,G,d,dv", [(4, 2, 128, 128), (3, 3, 64, 128), (2, 2, 128, 64), (5, 5, 64, 32), (2, 2, 32, 128), (2, 2, 64, 48)])
@pytest.mark.parametrize("B", [1, 3, 50])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_against_the_plain_form(gpu, mode, H, G, d, dv, B, dtype):
  """Sums of at most 128 products of unit-size numbers in fp32, another order: 128 * 2^-24 of the largest, and the decays' and gates'
  exponentials (a few 2^-24 each); bf16 results one rounding more.  The last two sizes run on the general kernels."""
  G = H if mode == "gla" else G
  a = inputs(mode, B, H, G, d, dv, B + d + dv)
  dev = {n: t.to(gpu) if torch.is_tensor(t) else t for n, t in a.items()}
  if a["gla"]:
    dev["gla"] = tuple(t.to(gpu) if torch.is_tensor(t) else t for t in a["gla"])
  out, got = torch.zeros(B, H * dv), torch.zeros(B, H * dv + 8, dtype=dtype, device=gpu)
  K.recurrence_norm(**a, out=out)
  K.recurrence_norm(**dev, out=got[:, :H * dv])
  torch.testing.assert_close(dev["state"].cpu(), a["state"], rtol=2e-5, atol=2e-5)
  live = a["state_slots"] >= 0
  rtol = 2 ** -8 if dtype == torch.bfloat16 else 1e-4
  torch.testing.assert_close(got[:, :H * dv].cpu().float()[live], out[live], rtol=rtol, atol=1e-4)
  assert not got[:, H * dv:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("mode,d", [("delta", 128), ("gla", 64), ("gla", 32)])
@pytest.mark.parametrize("F,tiles", [(48, True), (4, False), (200, False), (50, False), (1040, True)])
@pytest.mark.parametrize("B", [1, 37])
def test_activation_along_with_it(gpu, mode, d, F, tiles, B):
  """gelu(gate) * up in the same launch (columns apart, or alternating in tiles of 16; widths that are no multiple of four and
  uncovered key dims take a launch of its own): exactly gelu_mul's rows, and the recurrence's as without it."""
  H, dv = 2, 32
  a = inputs(mode, B, H, H, d, dv, B + F)
  dev = {n: t.to(gpu) if torch.is_tensor(t) else t for n, t in a.items()}
  if a["gla"]:
    dev["gla"] = tuple(t.to(gpu) if torch.is_tensor(t) else t for t in a["gla"])
  P = torch.randn(B, 8 + 2 * F + 32, device=gpu)
  args = (P, 8, -1, F) if tiles else (P, 8, 8 + F, F)
  want = torch.zeros(B, F + 8, dtype=torch.bfloat16, device=gpu)
  K.gelu_mul(*args, want)
  act, state = torch.zeros_like(want), dev["state"].clone()
  live = dev["state_slots"] >= 0  # (rows without a slot are not written)
  out, plain = (torch.zeros(B, H * dv, device=gpu) for _ in range(2))
  K.recurrence_norm(**dev, out=plain)
  K.recurrence_norm(**dict(dev, state=state), out=out, gelu=(*args, act))
  assert torch.equal(act, want) and torch.equal(out[live], plain[live]) and torch.equal(state, dev["state"])
