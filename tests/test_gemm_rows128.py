"""The 128- and 64-row tiles (and the 160 x 256 one) of the large-M GEMM (csrc/gemm_big.hip codes 1280128, 1280256, 640128, 640256): partial row and column tiles, fewer stages
than the pipeline holds, K splits, every epilogue; and where the policy offers them."""
import os
import subprocess
import sys

import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L
from xotorch_support_jetson_amd.ops.weights_layout import shuffle_for_stream


def test_candidates():
  """128-row tiles where they hold all rows, 128 x 128 up to 256 rows; no preference for half-empty 256-row tiles."""
  codes = lambda M: {c[1] for c in L.GemmPolicy._big_cands(M, 8192, 4096)}  # noqa: E731
  assert {1280128, 1280256} <= codes(65) and {1280128, 1280256} <= codes(128)
  assert 1280128 in codes(129) and 1280128 in codes(256) and 1280256 not in codes(129)
  assert 1280128 not in codes(257) and 1280128 not in codes(512)
  rows64 = L.GemmPolicy._rows64_cands
  assert {("big", 640128, 1), ("big", 640256, 8)} <= set(rows64(17, 8192, 4096)) and rows64(64, 128, 128) == [("big", 640128, 1)]
  assert rows64(16, 8192, 4096) == [] and rows64(65, 8192, 4096) == [] and rows64(64, 8200, 4096) == []
  times = {("big", 1280256, 1): 1.0, ("big", 2256, 1): 1.04}
  assert L._tie_break(times, 128) == ("big", 1280256, 1) and L._tie_break(times, 200) == ("big", 2256, 1)


@pytest.mark.parametrize("least,offered", [("129", [False] * 3), ("40", [False, True, True]), (None, [True] * 3)])
def test_switch_keeps_the_kernel_out(least, offered):
  """XOT_BIG_MIN_M holds for the 64-row tiles as well: rows 24, 40 and 64."""
  code = ("from xotorch_support_jetson_amd.ops import linear as L\n"
          "print([bool(L.GemmPolicy._rows64_cands(M, 8192, 4096)) for M in (24, 40, 64)])")
  env = {k: v for k, v in os.environ.items() if k != "XOT_BIG_MIN_M"}
  if least:
    env["XOT_BIG_MIN_M"] = least
  got = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, check=True)
  assert got.stdout.strip() == str(offered)


@pytest.mark.gpu
@pytest.mark.parametrize("code,M", [(c, m) for c, ms in ((1280128, (1, 65, 128, 129, 256)), (1280256, (1, 65, 128, 129)),
                                                         (640128, (1, 17, 63, 64, 65)), (640256, (1, 17, 63, 64, 65)), (1600256, (1, 160, 161, 320))) for m in ms])
@pytest.mark.parametrize("N,Kd,S", [(256, 128, 1), (400, 128, 1), (512, 1408, 1), (272, 1024, 3), (512, 512, 4)])
def test_exact(gpu, code, M, N, Kd, S):
  """Integer operands: sums bit for bit, fp32 and bf16, with bias and residual; gated pairs within one rounding (2^-8)."""
  from xotorch_support_jetson_amd.ops._ext import require
  C = require()
  g = torch.Generator().manual_seed(M + N + Kd)
  rn = lambda *s: torch.randint(-3, 4, s, generator=g).to(torch.bfloat16)  # noqa: E731
  x, w, b, r = rn(M, Kd), rn(N, Kd), rn(N), rn(M, N)
  full = x.float() @ w.float().t()
  xd, ws, ws_buf = x.to(gpu), shuffle_for_stream(w.to(gpu)), torch.empty(S * M * N, device=gpu)
  y = torch.empty(M, N, device=gpu)
  C.gemm_big(xd, ws, y, None, None, ws_buf, K.EPI["none"], code, S, True)
  assert torch.equal(y.cpu(), full)
  y = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
  C.gemm_big(xd, ws, y, b.to(gpu), r.to(gpu), ws_buf, K.EPI["resid"], code, S, True)
  assert torch.equal(y.cpu(), (full + b.float() + r.float()).to(torch.bfloat16))
  if N % 32 == 0:
    gate, up = (full.double().view(M, N // 32, 2, 16)[:, :, i].reshape(M, -1) for i in (0, 1))
    for epi, want in (("silu", gate * torch.sigmoid(gate) * up),
                      ("clamp_glu", gate.clamp(max=7) * torch.sigmoid(1.702 * gate.clamp(max=7)) * (up.clamp(-7, 7) + 1))):
      if epi == "clamp_glu" and code != 1280128:
        continue  # (the one it is built with)
      a = torch.empty(M, N // 2, dtype=torch.bfloat16, device=gpu)
      C.gemm_big(xd, ws, a, None, None, ws_buf, K.EPI[epi], code, S, True, 7.0)
      torch.testing.assert_close(a.cpu().double(), want, rtol=2 ** -7, atol=1e-6)


def test_routed_models_keep_their_candidates(monkeypatch):
  """Attention weights of models with routed experts: the candidates of 17 to 256 rows are those without the tiles above, under keys
  of their own."""
  seen = {}
  monkeypatch.setattr(L.policy, "_lookup", lambda key: None)
  monkeypatch.setattr(L.policy, "_no_tuning", lambda: True)
  monkeypatch.setattr(L.policy, "_heuristic", lambda M, N, cands: seen.setdefault("cands", cands) and cands[0])
  for M in (17, 64, 100, 200):
    for kept in (False, True):
      w = torch.empty(6144, 4096, dtype=torch.bfloat16, device="meta")
      if kept:
        L.keep_order(w)
      seen.clear()
      L.policy.shuffled_cfg(torch.empty(M, 4096, dtype=torch.bfloat16, device="meta"), w, None, None, "none", torch.bfloat16, "rope")
      new = [c for c in seen["cands"] if c[0] == "wave" or (c[0] == "big" and L.tile_rows(c[1]) in (64, 128))]
      assert bool(new) != kept
