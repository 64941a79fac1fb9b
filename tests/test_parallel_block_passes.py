"""The passes between the GEMMs of parallel blocks at the edges of their kernels: row widths of the register kernel, slabs,
vector widths, runs of eight tokens."""
import pytest
import torch

from xotorch_support_jetson_amd.models.transformer import StatePool
from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as ref


def rnd(*shape, seed=0):
  return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def near(got, want, dtype=torch.float32):
  # fp32: the sums' order (at most a few thousand terms of the row's scale); bf16: half a step (at most 2^-8 of the value) beside it,
  # against the unrounded fp32 result
  tol = 2e-5 if dtype == torch.float32 else 2.0 ** -8 + 2e-5
  assert bool(((got.cpu().float() - want.float()).abs() <= tol * want.float().abs() + 2e-5 * want.float().abs().max()).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,pad", [(4, 0), (1020, 4), (1024, 0), (1028, 0), (2048, 0), (4096, 0), (4100, 0), (8192, 0), (8196, 0),
                                   (1030, 2), (1024, 3)])
@pytest.mark.parametrize("S1,S2", [(1, 1), (1, 0), (0, 0), (5, 2), (2, 9)])
def test_residual_sum_of_slabs(dtype, D, pad, S1, S2):
  T, eps = 3, 1e-5
  ys = [rnd(S, T, D + pad, seed=S) if S else None for S in (S1, S2)]
  s = [rnd(D, seed=9), rnd(D, seed=10)]
  x, g = rnd(T, D, seed=1), torch.tensor([1.3])
  want_x, want = x.clone(), torch.zeros(T, D + pad)
  ref.resid_scale_norm(want_x, *[v for y, sc in zip(ys, s) for v in ((None, None) if y is None else (y.sum(0), sc))], g, eps, want)
  xd, out = x.cuda(), torch.full((T, D + pad), 3.0, dtype=dtype, device="cuda")
  args = [v for y, sc in zip(ys, s) for v in ((None, None) if y is None else ((y[0] if y.shape[0] == 1 else y).cuda(), sc.cuda()))]
  K.resid_scale_norm(xd, *args, gain=g.cuda(), eps=eps, out=out)
  near(xd, want_x)
  near(out[:, :D], want[:, :D], dtype)
  assert bool((out[:, D:] == 3.0).all())
  keep = xd.clone()
  K.resid_scale_norm(xd, *args, gain=None, eps=eps, out=None)  # the sum alone
  ref.resid_scale_norm(cpu := keep.cpu(), *[v.cpu().sum(0) if v is not None and v.dim() == 3 else v if v is None else v.cpu() for v in args],
                       None, eps, None)
  near(xd, cpu)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 9, 511, 512, 517])
@pytest.mark.parametrize("HD,rank,off", [(255, 1, 0), (256, 16, 4), (260, 5, 3), (1024, 256, 8), (64, 300, 0)])
def test_gla_decay(T, HD, rank, off):
  P, a2, b = rnd(T, off + rank + 2, seed=T), rnd(HD, rank, seed=2) / rank ** 0.5, rnd(HD, seed=3) + 2
  want = torch.empty(T, HD)
  ref.gla_prep(P, off, a2, b, 16.0, want)
  got = torch.empty(T, HD, device="cuda")
  K.gla_prep(P.cuda(), off, a2.cuda(), b.cuda(), 16.0, got)
  near(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,dv,off", [(1, 1, 0), (3, 64, 1), (5, 66, 2), (4, 128, 4), (4, 128, 1), (2, 130, 2), (6, 192, 4), (2, 256, 0),
                                      (3, 260, 8), (1, 515, 3)])
def test_gated_head_norm(dtype, H, dv, off):
  T = 3
  o, w, P = rnd(T, H * dv, seed=1), rnd(dv, seed=2), rnd(T, off + H * dv + 1, seed=3)
  P[0, off], o[1] = 90.0, 0.0  # a saturated gate, a row of zeros
  want, got = torch.zeros(T, H * dv), torch.zeros(T, H * dv, dtype=dtype, device="cuda")
  ref.gated_rmsnorm(o, w, P, off, 1e-5, 0.7, want)
  K.gated_rmsnorm(o.cuda(), w.cuda(), P.cuda(), off, 1e-5, 0.7, got)
  near(got, want, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,d,dv,taps", [(2, 1, 16, 24, 4), (4, 2, 128, 128, 4), (4, 4, 64, 130, 3), (2, 2, 256, 256, 4), (3, 1, 100, 30, 1),
                                           (2, 1, 8, 300, 6)])
@pytest.mark.parametrize("lens", [[1, 1, 1], [1], [3, 0, 70, 1], [300, 9]])
def test_delta_rule_inputs(H, G, d, dv, taps, lens):
  """Convolutions, gates and the carried inputs, one launch for single tokens (max_qlen 1) and in runs; a padding row changes
  no state."""
  C, T, B = 2 * G * d + H * dv, sum(lens), len(lens)
  cu = torch.tensor([0] + lens).cumsum(0).int()
  slots = torch.arange(B).flip(0).int()
  if B == 3:
    slots[1] = -1
  P, st = rnd(T, C + 2 * H + 3, seed=4), rnd(B + 1, taps - 1, C, seed=5)
  w, A, db = rnd(C, taps, seed=6), rnd(H, seed=7), rnd(H, seed=8)
  units, width = ref.conv_units(ref.delta_units(H, G, d, dv), C)
  live = torch.cat([torch.full((n,), int(s) >= 0) for n, s in zip(lens, slots)]) if T else torch.zeros(0, dtype=torch.bool)
  out = {}
  for dev in ("cpu", "cuda"):
    o = [torch.zeros(T, n, device=dev) for n in (C, H, H)]
    state = st.clone().to(dev)
    K.conv_prep(P.to(dev), 0, w.to(dev), None, units.to(dev), None, state, slots.to(dev), cu.to(dev), 0.0, o[0], max_qlen=max(lens),
                width=width, delta=(C, C + H, db.to(dev), A.to(dev), o[1], o[2]))
    out[dev] = [t[live.to(dev)] for t in o] + [state]
  for got, want in zip(out["cuda"], out["cpu"]):
    if want.numel():
      near(got, want)
  assert torch.equal(out["cuda"][3].cpu(), out["cpu"][3])  # (copies)


def test_slots_are_cleared_in_runs():
  class Pool(StatePool):
    def __init__(self, ts):
      self.S, self.conv, self.aux = ts[:1], ts[1:], [None]
  ts = [torch.ones(9, 2, 3), torch.ones(9, 4)]
  Pool(ts).clear([7, 2, 3, 0, 8])
  for t in ts:
    assert [int(r.abs().sum() > 0) for r in t] == [0, 1, 0, 0, 1, 1, 1, 0, 0]


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_delta_rule_inputs_of_an_empty_step(dev):
  H, G, d, dv, taps = 2, 1, 8, 16, 3
  C = 2 * G * d + H * dv
  e = lambda *s: torch.empty(*s, device=dev)  # noqa: E731
  state = torch.ones(1, taps - 1, C, device=dev)
  K.delta_prep(e(0, C + 2 * H), 0, C, C + H, e(C, taps), state, torch.empty(0, dtype=torch.int32, device=dev),
               torch.zeros(1, dtype=torch.int32, device=dev), e(H), e(H), H, G, d, dv, e(0, C), e(0, H), e(0, H))
  assert bool((state == 1).all())
