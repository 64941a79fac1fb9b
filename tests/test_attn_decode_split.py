"""Decode attention over units cut by the step's contexts: the plan's units, the merge inside the launch, and the rule that takes it."""
import math

import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R


def test_rule():
  assert not K.plan_pays(24, 8, 8) and K.plan_pays(24, 8, 9) and K.plan_pays(255, 8, 32)
  assert not K.plan_pays(256, 8, 32) and not K.plan_pays(128, 8, 16) and not K.plan_pays(256, 8, 4096)
  bt, cl = torch.zeros(24, 32, dtype=torch.int32), torch.zeros(24, dtype=torch.int32)
  assert K.DecodeWorkspace(24, 32, 128, 2048, torch.device("cpu")).plan(bt, cl, 8) is None  # (the plan is a kernel's)


def _step(lens, width, H, Hkv, Dh):
  g = torch.Generator(device="cuda").manual_seed(width + len(lens))
  pages = sum(-(-n // 64) for n in lens) + 1
  kc = torch.randn(pages, Hkv, 64, Dh, generator=g, device="cuda").bfloat16()
  vc = torch.randn(pages, Hkv, Dh, 64, generator=g, device="cuda").bfloat16()
  perm, at = torch.randperm(pages, generator=g, device="cuda").int().cpu(), 0
  bt = torch.zeros(len(lens), width, dtype=torch.int32)
  for i, n in enumerate(lens):
    m = -(-n // 64)
    bt[i, :m] = perm[at:at + m]
    at += m
  q = torch.randn(len(lens), H, Dh, generator=g, device="cuda").bfloat16()
  return q, kc, vc, bt.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda")


LENS = {"edges": [1, 63, 64, 65, 255, 256, 257, 320, 576, 0, 0], "one long": [17 * 64 + 3] + [40] * 6, "even": [900] * 12,
        "ragged": [int(70 * 20 ** (i / 23)) for i in range(24)], "one": [2000], "empty": [0, 0, 0], "many": [(7 * i) % 600 + 1 for i in range(515)]}


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hkv,Dh", [(32, 8, 128), (16, 1, 128), (14, 2, 64), (6, 6, 64)])
@pytest.mark.parametrize("lens", LENS)
def test_split_kernel(H, Hkv, Dh, lens):
  lens = LENS[lens]
  B, width = len(lens), max(9, -(-max(lens) // 64))
  q, kc, vc, bt, cl = _step(lens, width, H, Hkv, Dh)
  ws = K.DecodeWorkspace(B, H, Dh, width * 64, q.device, algo=2)
  C = K.require()
  plan = C.decode_plan(cl, B, Hkv, width)
  rows = [r for r in plan.tolist() if r[3]]
  at = 0
  for b, n in enumerate(lens):  # a sequence's parts: one behind the other, equal to a page, together all of its pages
    pages, mine = -(-n // 64), rows[at:at + rows[at][3]]
    assert [r[0] for r in mine] == [b] * len(mine) and all(r[3:6] == [len(mine), at, n] for r in mine)
    assert mine[0][1] == 0 and mine[-1][2] == pages and all(x[2] == y[1] for x, y in zip(mine, mine[1:]))
    sizes = [r[2] - r[1] for r in mine]
    assert max(sizes) - min(sizes) <= 1 and (len(mine) == 1 or min(sizes) >= 2)
    at += len(mine)
  assert at == len(rows)
  live = [i for i, n in enumerate(lens) if n]
  runs = []
  for nt in (False, True, False):
    out = torch.full_like(q, float("nan"))
    C.attn_decode_split(q, kc, vc, bt, plan, cl, ws.tickets, out, ws.o, ws.ml, Dh ** -0.5, nt)
    assert int(ws.tickets.abs().max()) == 0
    runs.append(out)
  assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])  # whoever merges, in the order of the parts
  assert all(float(runs[0][i].abs().max()) == 0.0 for i, n in enumerate(lens) if not n)
  if live:
    want = R.attn_decode(q[live], kc, vc, bt[live], cl[live], 1 / math.sqrt(Dh)).float()
    # probabilities and results in bf16 (2^-9 each, of values at most a few): as for the other decode kernels
    assert float((runs[0][live].float() - want).abs().max()) < 2e-2 * float(want.abs().max())


@pytest.mark.gpu
def test_plan_follows_the_contexts_under_a_graph():
  """One captured step serves contexts of any length: plan and attention replayed with other lengths, against an eager step."""
  H, Hkv, Dh, width = 32, 8, 128, 32
  lens = LENS["ragged"]
  q, kc, vc, bt, cl = _step(lens, width, H, Hkv, Dh)
  ws = K.DecodeWorkspace(len(lens), H, Dh, width * 64, q.device)

  def step():
    plan = ws.plan(bt, cl, Hkv)
    assert plan is not None
    return K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws, plan=plan)
  side = torch.cuda.Stream()
  side.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(side):
    step()
  torch.cuda.current_stream().wait_stream(side)
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    got = step()
  for cut in (1, 3, 50, 2):
    cl.copy_(torch.tensor([max(1, n // cut) for n in lens], dtype=torch.int32))
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(got, step())
    whole = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, K.DecodeWorkspace(len(lens), H, Dh, width * 64, q.device, pages_per_part=width, algo=2))
    assert float((got.float() - whole.float()).abs().max()) < 2e-2 * float(whole.float().abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hkv,Dh", [(32, 8, 64), (16, 1, 128), (14, 2, 64), (32, 32, 128)])
def test_lone_sequence_needs_no_plan(H, Hkv, Dh):
  for width in (1, 8, 40, 128):
    ws = None
    for n in sorted({1, 64, 65, 255, 257, 321, width * 64 - 1, width * 64, 0} & set(range(width * 64 + 1))):
      q, kc, vc, bt, cl = _step([n], width, H, Hkv, Dh)
      ws = ws or K.DecodeWorkspace(1, H, Dh, width * 64, q.device)
      assert ws.plan(bt, cl, Hkv) is K.LONE
      out = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws, plan=K.LONE)
      assert torch.equal(out, K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws, plan=K.LONE)) and int(ws.tickets.abs().max()) == 0
      if n == 0:
        assert float(out.abs().max()) == 0.0
        continue
      want = R.attn_decode(q, kc, vc, bt, cl, 1 / math.sqrt(Dh)).float()
      # (as above)
      assert float((out.float() - want).abs().max()) < 2e-2 * float(want.abs().max()), (width, n)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,Hkv,Dh,whole", [([600] * 40, 8, 128, True), ([300] * 150, 2, 64, True), ([1000] * 100, 16, 128, True), ([1600] + [100] * 23, 8, 128, False),
                                               ([3000] * 4, 8, 64, False), ([17 * (i + 1) for i in range(40)], 8, 64, True)])
def test_contexts_that_fill_the_chip_stay_whole(lens, Hkv, Dh, whole):
  """A merge costs about four pages, of heads of 64 seven, which a cut has to bring in."""
  cl = torch.tensor(lens, dtype=torch.int32, device="cuda")
  parts = K.require().decode_plan(cl, len(lens), Hkv, 64, Dh)[:, 3].max().item()
  assert (parts == 1) == whole


@pytest.mark.gpu
def test_steps_too_large_to_count_are_refused():
  """Pages over all KV heads are counted in 32 bits, and a plan belongs to the batch and the tables it was made for."""
  C = K.require()
  cl = torch.ones(1 << 20, dtype=torch.int32, device="cuda")
  for B, Hkv, width in ((1, 1 << 10, 1 << 20), (1 << 20, 1 << 10, 1), (1 << 20, 1 << 4, 1), (1 << 15, 1 << 5, 1 << 10), (1 << 10, 1 << 20, 1 << 24), (1, 1, (1 << 24) + 1), (0, 8, 9), (2, 0, 9)):
    with pytest.raises(RuntimeError):
      C.decode_plan(cl, B, Hkv, width)
  q, kc, vc, bt, cl = _step([600] * 6, 10, 16, 4, 64)
  ws = K.DecodeWorkspace(64, 16, 64, 64 * 64, q.device, algo=2)
  for B, width in ((5, 10), (7, 10), (64, 64)):  # (no plan of these has as many places)
    plan = C.decode_plan(torch.full((B,), 600, dtype=torch.int32, device="cuda"), B, 4, width)
    with pytest.raises(RuntimeError):
      C.attn_decode_split(q, kc, vc, bt, plan, cl, ws.tickets, torch.empty_like(q), ws.o, ws.ml, 0.125, False)
  assert int(ws.tickets.abs().max()) == 0


def test_places_of_the_rule():
  """Every plan of a workspace's own batches and widths fits it (a KV head has at most 16 query heads)."""
  for max_batch, H, max_ctx in ((1, 32, 300), (4, 64, 2048), (32, 32, 512), (300, 14, 9000)):
    ws = K.DecodeWorkspace(max_batch, H, 128, max_ctx, torch.device("cpu"))
    for Hkv in (n for n in range(1, H + 1) if H % n == 0 and H // n <= 16):
      assert all(K.split_places(B, Hkv, w) <= ws.places for B in {1, max_batch // 2 or 1, max_batch} for w in range(1, -(-max_ctx // 64) + 1))


@pytest.mark.gpu
def test_tables_wider_than_the_workspace():
  """A workspace of a shorter context bound serves wide tables as it can: whole contexts, no plan."""
  B, H, Hkv, Dh, width = 32, 16, 8, 128, 32
  q, kc, vc, bt, cl = _step([40 + (53 * i) % 1100 for i in range(B)], width, H, Hkv, Dh)
  ws = K.DecodeWorkspace(B, H, Dh, 512, q.device)
  plan = ws.plan(bt, cl, Hkv)
  out = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws, plan=plan)
  want = R.attn_decode(q, kc, vc, bt, cl, 1 / math.sqrt(Dh)).float()
  assert float((out.float() - want).abs().max()) < 2e-2 * float(want.abs().max())  # (as above)
  assert plan is None and K.DecodeWorkspace(B, H, Dh, width * 64, q.device).plan(bt, cl, Hkv) is not None
  assert K.split_places(7, Hkv, 33) == K.require().decode_plan(cl.new_ones(7), 7, Hkv, 33).shape[0]
