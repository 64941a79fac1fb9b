"""Prompts of unlike lengths in one step: every workgroup of the launch finds its sequence, head and rows, whatever the batch."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R

# (new tokens, cached tokens) per sequence: one, two equal ones, a pair count that is no multiple of 8, the sorted range's end and past it
BATCHES = {"one": [(300, 0)], "equal": [(64, 0)] * 2, "decode and prompt": [(1, 700), (500, 0), (1, 30)], "nine": [(7 + 67 * (4 * i % 9), 31 * i) for i in range(9)],
           "32": [(1 + 37 * i % 211, 0) for i in range(32)], "33": [(1 + 37 * i % 211, 0) for i in range(33)]}


def _step(batch, G, d):
  g = torch.Generator(device="cuda").manual_seed(len(batch) + G)
  ctx = [n + m for n, m in batch]
  width, pages = max(-(-c // 64) for c in ctx), sum(-(-c // 64) for c in ctx)
  kc = torch.randn(pages, G, 64, d, generator=g, device="cuda").bfloat16()
  vc = torch.randn(pages, G, d, 64, generator=g, device="cuda").bfloat16()
  perm, bt, at = torch.randperm(pages, generator=g, device="cuda").int().cpu(), torch.zeros(len(ctx), width, dtype=torch.int32), 0
  for b, c in enumerate(ctx):
    bt[b, :-(-c // 64)] = perm[at:at - (-c // 64)]
    at += -(-c // 64)
  cu = torch.tensor([0] + [n for n, _ in batch]).cumsum(0).int().cuda()
  return kc, vc, bt.cuda(), cu, torch.tensor(ctx, dtype=torch.int32, device="cuda"), g


# bf16 probabilities (2^-9 each, independent) and a bf16 result (2^-9): well within 2^-6 of the largest value
def _near(y, ref):
  assert (y.float() - ref.float()).abs().max() <= 2**-6 * ref.float().abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("H,G", [(32, 8), (6, 3), (4, 4)])
@pytest.mark.parametrize("batch", BATCHES)
def test_causal(batch, H, G):
  batch = BATCHES[batch]
  kc, vc, bt, cu, cl, g = _step(batch, G, 128)
  q = torch.randn(sum(n for n, _ in batch), H, 128, generator=g, device="cuda").bfloat16()
  args = (q, kc, vc, bt, cu, cl)
  out = torch.full_like(q, float("nan"))
  K.attn_prefill(*args, max(n for n, _ in batch), 128**-0.5, out=out)
  _near(out, R.attn_prefill(*args, 128**-0.5))


@pytest.mark.gpu
@pytest.mark.parametrize("H,G", [(16, 4), (6, 3), (8, 8)])
@pytest.mark.parametrize("batch", BATCHES)
def test_window(batch, H, G):
  batch = BATCHES[batch]
  kc, vc, bt, cu, cl, g = _step(batch, G, 128)
  q = torch.randn(sum(n for n, _ in batch), H, 128, generator=g, device="cuda").bfloat16()
  args, longest = (q, kc, vc, None, None, bt, cu, cl), max(n for n, _ in batch)
  out, ref = torch.full((len(q), H * 128), float("nan"), device="cuda"), torch.zeros(len(q), H * 128)
  K.attn_window_pool(*args, None, 128**-0.5, 200, 0, out, longest, 0, 4)
  R.attn_window_pool(*(x if x is None else x.cpu() for x in args), None, 128**-0.5, 200, 0, ref, longest, 0, 4)
  _near(out.cpu(), ref)


# a workgroup's arithmetic does not know the batch: each sequence as it comes alone (which other tests hold against float64)
@pytest.mark.gpu
@pytest.mark.parametrize("B", [2, 5, 7, 8, 9, 32, 33])  # 64 workgroups a sequence: up to 256, up to 512, and more; sorted and as given
def test_scan_alone(B):
  H, G, d, dv = 16, 4, 64, 128
  lens = [64 + 53 * (5 * i % B) % 190 for i in range(B)]
  g = torch.Generator(device="cuda").manual_seed(B)
  rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
  T, cu = sum(lens), torch.tensor([0] + lens).cumsum(0).int().cuda()
  q, k, v = rn(T, G * d) / 8, rn(T, G * d) / 8, rn(T, H * dv)
  decay, beta, state = torch.sigmoid(rn(T, H) + 3), torch.sigmoid(rn(T, H)), rn(B, H, dv, d)
  slots, S, out = torch.randperm(B, generator=g, device="cuda").int(), state.clone(), torch.full((T, H * dv), float("nan"), device="cuda")
  K.linear_recurrence(q, k, v, decay, beta, 0.5, S, slots, cu, out, False, max(lens))
  for b, n in enumerate(lens):
    rows, one = slice(int(cu[b]), int(cu[b]) + n), torch.empty(n, H * dv, device="cuda")
    K.linear_recurrence(q[rows], k[rows], v[rows], decay[rows], beta[rows], 0.5, state, slots[b:b + 1], torch.tensor([0, n]).int().cuda(), one,
                        False, max(lens))
    assert torch.equal(one, out[rows]), b
  assert torch.equal(state, S)


@pytest.mark.gpu
def test_scan_of_many_workgroups():
  """More workgroups than one launch dimension holds work items for, all but two sequences' without tokens: the last one runs too."""
  B, H, d, dv, n = 32769, 16, 64, 1024, 97  # x 32 column blocks: 2^24 + 512
  g = torch.Generator(device="cuda").manual_seed(3)
  rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
  q, k, v = rn(2 * n, H * d) / 8, rn(2 * n, H * d) / 8, rn(2 * n, H * dv)
  decay, beta, state = torch.sigmoid(rn(2 * n, H) + 3), torch.sigmoid(rn(2 * n, H)), rn(2, H, dv, d)
  cu, slots = torch.full((B + 1,), n, dtype=torch.int32), torch.full((B,), -1, dtype=torch.int32)
  cu[0], cu[-1], slots[0], slots[-1] = 0, 2 * n, 0, 1
  S, out, one = state.clone(), torch.full((2 * n, H * dv), float("nan"), device="cuda"), torch.empty(2 * n, H * dv, device="cuda")
  K.linear_recurrence(q, k, v, decay, beta, 0.5, S, slots.cuda(), cu.cuda(), out, False, n)
  K.linear_recurrence(q, k, v, decay, beta, 0.5, state, torch.tensor([0, 1]).int().cuda(), torch.tensor([0, n, 2 * n]).int().cuda(), one, False, n)
  assert torch.equal(out, one) and torch.equal(S, state)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G", [(16, 4), (6, 3)])
@pytest.mark.parametrize("batch", BATCHES)
def test_gated_alone(batch, H, G):
  batch = BATCHES[batch]
  kc, vc, bt, cu, cl, g = _step(batch, G, 64)
  q, pb = torch.randn(int(cu[-1]), H, 64, generator=g, device="cuda").bfloat16(), torch.randn(H, generator=g, device="cuda")
  out = torch.full((len(q), H * 64), float("nan"), device="cuda", dtype=torch.bfloat16)
  K.attn_gated_chunk(q, kc, vc, bt, cu, cl, pb, 0.125, 256, 0.5, out, max(n for n, _ in batch))
  for b, (n, _) in enumerate(batch):
    rows = slice(int(cu[b]), int(cu[b]) + n)
    one = torch.empty(n, H * 64, device="cuda", dtype=torch.bfloat16)
    K.attn_gated_chunk(q[rows], kc, vc, bt[b:b + 1], torch.tensor([0, n]).int().cuda(), cl[b:b + 1], pb, 0.125, 256, 0.5, one, max(n, 2))
    assert torch.equal(one, out[rows]), b


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,longest", [(5, 52, 65535 * 128), (66000, 2, 2)])
def test_gated_chunk_of_many_workgroups(B, H, longest):
  """More workgroups than one launch dimension holds work items for, most of them without rows (the longest run is a bound), and a
  large batch: what the launch is told does not change the rows."""
  d, T = 32, B + 4
  g = torch.Generator(device="cuda").manual_seed(H)
  kc, vc = (torch.randn(1, 1, *s, generator=g, device="cuda").bfloat16() for s in ((64, d), (d, 64)))
  q = torch.randn(T, H, d, generator=g, device="cuda").bfloat16()
  pb, cu = torch.randn(H, generator=g, device="cuda"), torch.arange(B + 1, dtype=torch.int32, device="cuda")
  cu[-1] = T  # the last sequence has five tokens, the others one
  cl = torch.ones(B, dtype=torch.int32, device="cuda")
  cl[-1] = 5
  bt = torch.zeros(B, 1, dtype=torch.int32, device="cuda")
  out = torch.full((T, H * d), float("nan"), device="cuda", dtype=torch.bfloat16)
  K.attn_gated_chunk(q, kc, vc, bt, cu, cl, pb, d**-0.5, 1024, 1.0, out, longest)
  torch.cuda.synchronize()
  k, v = kc[0, 0, :5].double(), vc[0, 0, :, :5].t().double()
  w = torch.sigmoid(q.double() @ k.t() * d**-0.5 + pb.double()[:, None])
  pos = torch.cat([torch.zeros(B - 1, dtype=torch.long), torch.arange(5)]).cuda()
  w = w * (torch.arange(5, device="cuda") <= pos[:, None])[:, None]
  _near(out, (w @ v).reshape(T, H * d))
