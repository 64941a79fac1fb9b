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


def float64_rows(a):
  """recurrence_norm's definition in float64, token by token (inputs' single tokens), and the rows that have a slot."""
  B, (_, H, dv, d) = a["q"].shape[0], a["state"].shape
  G = a["q"].shape[1] // d
  q, k, v, w, gate = (a[n].double() for n in ("q", "k", "v", "w", "gate"))
  heads = lambda t: t.reshape(B, G, d).repeat_interleave(H // G, 1)  # noqa: E731
  q, k, v = heads(q) * a["q_scale"], heads(k), v.reshape(B, H, dv)
  S = a["state"].double()[a["state_slots"].clamp(min=0).long()]
  if a["beta"] is None:
    P, c0, a2, b, tau = a["gla"]
    decay = torch.exp(torch.nn.functional.logsigmoid(P[:, c0:c0 + a2.shape[1]].double() @ a2.double().t() + b.double()) / tau)
  else:
    decay = a["decay"].double()
  S = S * decay.reshape(B, H, 1, -1)
  u = v if a["beta"] is None else a["beta"].double()[..., None] * (v - torch.einsum("bhvd,bhd->bhv", S, k))
  o = torch.einsum("bhvd,bhd->bhv", S + u[..., None] * k[:, :, None], q)
  gate = gate[:, :H * dv].reshape(B, H, dv)
  o = o / torch.sqrt(o.square().mean(-1, keepdim=True) + a["eps"]) * (w.view(H, dv) if w.numel() == H * dv else w)
  o = o * (torch.sigmoid(gate) if a["sigmoid"] else torch.nn.functional.silu(gate)) * a["scale"]
  return o.reshape(B, H * dv), a["state_slots"] >= 0


def norm_forms(mode, sigmoid, per_head, d, B=5):
  H, G, dv = 4, 4 if mode == "gla" else 2, 64
  a = inputs(mode, B, H, G, d, dv, d + 7)
  w = torch.randn(H * dv if per_head else dv, generator=torch.Generator().manual_seed(3))
  return dict(a, sigmoid=sigmoid, scale=0.7, w=w), torch.zeros(B, H * dv)


@pytest.mark.parametrize("mode", ["delta", "channel", "gla"])
@pytest.mark.parametrize("sigmoid", [False, True])
@pytest.mark.parametrize("per_head", [False, True])
def test_every_norm_form_means_the_same(mode, sigmoid, per_head):
  """Both gates with both weights and a scale, by the passes behind each other."""
  a, out = norm_forms(mode, sigmoid, per_head, 64)
  want, live = float64_rows(a)
  K.recurrence_norm(**a, out=out)
  torch.testing.assert_close(out[live].double(), want[live], rtol=1e-4, atol=1e-4)  # (bound: test_against_the_plain_form)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["delta", "channel", "gla"])
@pytest.mark.parametrize("sigmoid", [False, True])
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("d,max_qlen", [(64, 1), (64, 0), (32, 1)])
def test_every_norm_form_on_every_route(gpu, mode, sigmoid, per_head, d, max_qlen):
  """The same on the GPU: in one launch, and by general kernels where the step's longest sequence is not known or the key
  dims are not covered."""
  a, out = norm_forms(mode, sigmoid, per_head, d)
  want, live = float64_rows(a)
  dev = {n: t.to(gpu) if torch.is_tensor(t) else t for n, t in a.items()}
  if a["gla"]:
    dev["gla"] = tuple(t.to(gpu) if torch.is_tensor(t) else t for t in a["gla"])
  out = out.to(gpu)
  K.recurrence_norm(**dict(dev, max_qlen=max_qlen), out=out)
  torch.testing.assert_close(out.cpu()[live].double(), want[live], rtol=1e-4, atol=1e-4)
