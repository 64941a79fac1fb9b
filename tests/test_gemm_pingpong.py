"""The ping-pong schedules of csrc/gemm_big.hip, two-phase (tile codes 2256 / 2192 / 2128) and four-phase (1256): their order of LDS reads
and refills, on a model of the workgroup's barriers, and the former's products at few k stages."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops.weights_layout import shuffle_for_stream


def former(t, T):
  """A stage as it once was: the whole refill behind this wave's own reads of A half 1, the first reads not waited for."""
  yield from (("read", "A0"), ("read", "B"), "bar", "lgkm", "bar", ("read", "A1"), "lgkm")
  if t + 2 < T:
    yield from (("issue", "A0", t + 2), ("issue", "B", t + 2), ("issue", "A1", t + 2))
  yield from (("landed", "A0", t + 1), ("landed", "B", t + 1), ("landed", "A1", t + 1), "bar", "lgkm", "bar")


def two_phase(t, T):
  """A stage of the kernel: one wave's reads, refills and waits (a wait: the refills that have landed behind it) in order."""
  yield from (("read", "B"), ("read", "A0"))
  if 0 < t < T - 1:
    yield ("issue", "A1", t + 1)
  if t > 0:
    yield ("landed", "A1", t)
  yield from ("lgkm B", "bar", "lgkm", "bar", ("read", "A1"))
  if t + 2 < T:
    yield from (("issue", "A0", t + 2), ("issue", "B", t + 2))
  yield from (("landed", "A0", t + 1), ("landed", "B", t + 1), "bar", "lgkm", "bar")


def four_phase(t, T):
  """A stage of the four-phase schedule (B's halves apart): everything is refilled in the last phase."""
  yield from (("read", "A0"), ("read", "B"), "bar", "lgkm", "bar", ("read", "B"), "bar", "lgkm", "bar", ("read", "A1"), "bar", "lgkm", "bar")
  if t + 2 < T:
    yield from (("issue", "A0", t + 2), ("issue", "B", t + 2), ("issue", "A1", t + 2))
  yield from (("landed", "A0", t + 1), ("landed", "B", t + 1), ("landed", "A1", t + 1), "bar", "bar")


def accesses(stage, T, half, wave):
  """[(wave, first barrier count, last barrier count, order, kind, LDS region, stage)] of one wave; a wave of row half 1 passes
  one barrier more before its first stage.  X rows are a half's own, W rows are everyone's."""
  at, out, reading, flying = 1 + half, [], [], {}
  for part in ("A0", "B", "A1"):  # the prologue: stage 0 has landed in front of the first barrier, stage 1 is on its way
    out.append((wave, -1, 0, -1, "write", (0, part, half), 0))
    if T > 1:
      flying[part, 1] = (0, -1)
  for t in range(T):
    for n, op in enumerate(stage(t, T)):
      if op == "bar":
        at += 1
      elif op in ("lgkm", "lgkm B"):  # (LDS reads return in order: those of B come first)
        out += [(wave, a, at, k, "read", r, s) for a, k, r, s in reading if op == "lgkm" or r[1] == "B"]
        reading = [] if op == "lgkm" else [r for r in reading if r[2][1] != "B"]
      elif op[0] == "read":
        reading.append((at, (t, n), (t % 2, op[1], half), t))
      elif op[0] == "issue":
        flying[op[1], op[2]] = (at, (t, n))
      elif (op[1], op[2]) in flying:
        a, k = flying.pop((op[1], op[2]))
        out.append((wave, a, at, k, "write", (op[2] % 2, op[1], half), op[2]))
  assert not reading and not flying
  return out


def unordered(stage, T):
  """Pairs (read of stage s, refill) of different waves in one LDS region that no barrier puts in order, or in the wrong one."""
  every = [a for w in range(4) for a in accesses(stage, T, w // 2, w)]
  bad = []
  for r in every:
    for w in every:
      same = r[5] == w[5] if r[5][1] != "B" else r[5][:2] == w[5][:2]
      if r[4] != "read" or w[4] != "write" or not same or r[0] == w[0]:
        continue
      # (an access that ends at barrier count n is behind the others' accesses that start at n + 1)
      if not (w[2] < r[1] if w[6] <= r[6] else r[2] < w[1]):
        bad.append((r, w))
  return bad


def test_every_refill_is_a_barrier_away_from_its_readers():
  for T in range(1, 7):
    assert not unordered(two_phase, T) and not unordered(four_phase, T), T
  found = {(r[5][1], r[0] // 2 == w[0] // 2) for r, w in unordered(former, 5)}
  assert found == {("A1", True), ("B", False)}  # a half's own second rows; the other half's reads of W


def integers(gen, *shape):
  return torch.randint(-3, 4, shape, generator=gen).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("code", [2256, 1922256])
@pytest.mark.parametrize("Kd,S", [(128, 2), (128, 1), (384, 2), (256, 1), (640, 2), (384, 1), (1408, 1)])
def test_products_of_few_stages(gpu, code, Kd, S):
  """1 to 22 k stages, rows and columns past a tile, bit for bit on integers."""
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(Kd + S)
  M, N = 300, 528
  x, w = integers(g, M, Kd), integers(g, N, Kd)
  y, ws = torch.zeros(M, N, device=gpu), torch.zeros(S * M * N, device=gpu)
  require().gemm_big(x.to(gpu), shuffle_for_stream(w.to(gpu)), y, None, None, ws if S > 1 else None, K.EPI["none"], code, S, True)
  assert torch.equal(y.cpu(), x.float() @ w.float().t())


@pytest.mark.gpu
@pytest.mark.parametrize("bm", [2128, 2192, 2256])
@pytest.mark.parametrize("Kd,S", [(128, 2), (128, 1), (384, 2), (256, 1), (640, 2), (384, 1), (1408, 1)])
def test_experts_of_few_stages(gpu, bm, Kd, S):
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(Kd + S + bm)
  E, T, N = 5, 290, 512
  cnt = torch.tensor([T, 0, 17, 200, 1])
  off = torch.cat([torch.zeros(1, dtype=torch.long), cnt.cumsum(0)]).int()
  tok = torch.cat([torch.randperm(T, generator=g)[:c] for c in cnt]).int()
  x, w = integers(g, T, Kd), integers(g, E, N, Kd)
  y = torch.zeros(S * len(tok), N, device=gpu)
  require().gemm_moe(x.to(gpu), torch.stack([shuffle_for_stream(m.to(gpu)) for m in w]), y, off.to(gpu), tok.to(gpu), K.EPI["none"], T, True, S, bm)
  want = torch.cat([x[tok[off[e]:off[e + 1]].long()].float() @ w[e].float().t() for e in range(E)])
  assert torch.equal(y.view(S, -1, N).sum(0).cpu(), want)
