"""Latent attention in partitions of a few pages: parts past a sequence's end, more parts than a wave has lanes, every place of the launch."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import reference as R


@pytest.mark.parametrize("max_tokens,H,max_ctx", [(1, 16, 17 * 64), (1, 16, 4096), (37, 16, 2048), (512, 16, 4096), (8, 128, 8192), (3, 200, 1100), (1, 128, 8192),
                                                  (1, 16, 64000)])
def test_workspace_holds_every_table(max_tokens, H, max_ctx):
  ws = K.MLAWorkspace(max_tokens, H, 256, max_ctx, torch.device("cpu"))
  for width in [*range(1, ws.pages + 1), 2 * ws.pages, 100 * ws.pages]:
    for T in {1, 2, 3, 7, 8, 9, 100, 129, 255, 256, 300, max_tokens}:
      ppp, nparts, _ = ws.partition(T, width)
      assert ppp * nparts >= width > ppp * (nparts - 1)
      assert nparts == 1 or ws.o.numel() >= T * nparts * H * 256 and ws.ml.numel() >= T * nparts * H * 2


@pytest.mark.parametrize("H", [16, 32, 128])
def test_contexts_alike_are_one_round(H):
  """A part a CU, and one round of them where the CUs are enough; short tables and a prompt's rows that fill the chip stay whole."""
  ws = K.MLAWorkspace(64, H, 256, 4096, torch.device("cpu"))
  for T in range(1, 400):
    units = T * -(-H // 128) if ws.wide(T) else T * H // 16
    for width in (1, 2, 3, 4, 8, 16, 17, 40, 64):
      nparts = ws.partition(T, width)[1]
      assert nparts == 1 or units * nparts < 256 + units
      assert nparts == 1 or units <= 128 or width > 16 and T <= 64
      assert nparts == 1 or width > 3 or ws.wide(T)


# (contexts, new tokens, pages a part)
STEPS = {"ragged": ([1, 64, 65, 300, 0, 129, 700, 2], None, 1), "70 parts": ([70 * 64, 100, 65 * 64], None, 1), "37": ([20 + 41 * i % 500 for i in range(37)], None, 2),
         "prompts": ([130, 5, 200], [130, 1, 77], 2), "whole": ([130, 90], [130, 20], 8)}


@pytest.mark.gpu
@pytest.mark.parametrize("H,DL,wide", [(16, 512, False), (40, 256, False), (40, 512, True)])
@pytest.mark.parametrize("step", STEPS)
def test_parts(step, H, DL, wide, monkeypatch):
  ctxs, new, ppp = STEPS[step]
  new = new or [1] * len(ctxs)
  B, T, width = len(ctxs), sum(new), -(-max(ctxs) // 64)
  g = torch.Generator().manual_seed(B + H)
  rn = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
  q_lat, q_pe, cache = rn(H, T, DL), rn(T, H * 64), rn(B * width, 64, DL + 64)
  bt = torch.randperm(B * width, generator=g).int().view(B, width)
  cu, ctx = torch.tensor([0] + new).cumsum(0).int(), torch.tensor(ctxs).int()
  args = (q_lat, q_pe, cache, bt, cu, ctx)
  ref = R.mla_attn(*args, 0.04).float()
  monkeypatch.setattr(K.MLAWorkspace, "partition", lambda self, T, w: (ppp, -(-w // ppp), wide))
  out = K.mla_attn(*(x.cuda() for x in args), 0.04).float().cpu()
  rows = [t for b in range(B) for t in range(int(cu[b]), int(cu[b + 1])) if ctxs[b]]
  # bf16 probabilities and results, 2^-9 each of a row's values
  assert (out - ref)[:, rows].abs().max() <= 2**-6 * ref[:, rows].abs().max()
  assert not out[:, [t for t in range(T) if t not in rows]].any()


@pytest.mark.gpu
@pytest.mark.parametrize("H", [16, 40])
@pytest.mark.parametrize("lens", ["alike", "ragged", "64", "edge"])
def test_parts_by_the_contexts(H, lens):
  """Parts of two lengths, of which the step's contexts take one: both against the reference, whatever the batch leaves of a wave."""
  lens = {"alike": [900] * 37, "ragged": [62 + 22 * i for i in range(36)] + [0], "64": [(97 * i) % 1024 + 1 for i in range(64)],
          "edge": [1024] * 32}[lens]
  B, DL, width = len(lens), 256, 16
  g = torch.Generator().manual_seed(B + H)
  rn = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
  q_lat, q_pe, cache = rn(H, B, DL), rn(B, H * 64), rn(B * width, 64, DL + 64)
  bt = torch.randperm(B * width, generator=g).int().view(B, width)
  args = (q_lat, q_pe, cache, bt, torch.arange(B + 1).int(), torch.tensor(lens).int())
  ws = K.MLAWorkspace(B, H, DL, width * 64, torch.device("cuda"))
  ref = R.mla_attn(*args, 0.04).float()
  ws.o.fill_(float("nan"))
  ws.ml.fill_(float("nan"))
  out = K.mla_attn(*(x.cuda() for x in args), 0.04, ws).float().cpu()
  live = [b for b in range(B) if lens[b]]
  # bf16 probabilities and results, 2^-9 each of a row's values
  assert (out - ref)[:, live].abs().max() <= 2**-6 * ref[:, live].abs().max()
  assert not out[:, [b for b in range(B) if not lens[b]]].any()
