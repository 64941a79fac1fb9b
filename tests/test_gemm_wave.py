"""The whole-K decode GEMM (csrc/gemm_wave.hip): every epilogue, column width and prologue at the edges of its range."""
import pathlib
import re

import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L
from xotorch_support_jetson_amd.ops.weights_layout import shuffle_for_stream


def integers(gen, *shape):
  return torch.randint(-3, 4, shape, generator=gen).to(torch.bfloat16)


def test_candidates_cover_their_range_only():
  """Up to WAVE_MAX_M rows, whole column tiles, gate / up pairs inside a workgroup, one width for rotation pairs."""
  cands = L.GemmPolicy._wave_cands
  assert cands(1, 48, 128, "none", False) == [("wave", 1, 1)]
  assert cands(L.WAVE_MAX_M, 64, 128, "none", False) == [("wave", 1, 1), ("wave", 2, 1), ("wave", 4, 1)]
  assert cands(3, 64, 256, "silu", False) == [("wave", 2, 1), ("wave", 4, 1)]
  assert cands(3, 64, 256, "none", True) == [("wave", 2, 1)]
  assert cands(L.WAVE_MAX_M + 1, 64, 128, "none", False) == [] and cands(1, 64, 96, "none", False) == []


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 15, 16])
@pytest.mark.parametrize("N,Kd", [(64, 128), (192, 256), (320, 1408), (128, 4096)])
def test_epilogues_exact(gpu, M, N, Kd):
  """Integer operands: sums bit for bit (waves without a k block, uneven shares, a last stage that is not full), fp32 and bf16,
  bias, residual in place, relu^2, gated pairs, rows of a wider buffer."""
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(M + N + Kd)
  x, w, b, r = integers(g, M, Kd), integers(g, N, Kd), integers(g, N), integers(g, M, N)
  full = x.float() @ w.float().t()
  ws, bd, C = shuffle_for_stream(w.to(gpu)), b.to(gpu), require()
  wide = torch.zeros(M, Kd + 16, dtype=torch.bfloat16, device=gpu)
  wide[:, 8:8 + Kd] = x.to(gpu)
  xd = wide[:, 8:8 + Kd]
  for nt in (1, 2, 4):
    y = torch.zeros(M, N, device=gpu)
    C.gemm_wave(xd, ws, y, bd, None, K.EPI["none"], nt)
    assert torch.equal(y.cpu(), full + b.float()), nt
    h = r.to(gpu)
    C.gemm_wave(xd, ws, h, None, h, K.EPI["resid"], nt)
    assert torch.equal(h.cpu(), (full + r.float()).to(torch.bfloat16)), nt
    a = torch.zeros(M, N, dtype=torch.bfloat16, device=gpu)
    C.gemm_wave(xd, ws, a, None, None, K.EPI["relu2"], nt)
    assert torch.equal(a.cpu(), full.clamp(min=0).square().to(torch.bfloat16)), nt
    if nt == 1:
      continue
    f = (full + b.float()).view(M, N // 32, 2, 16)
    want = {"silu": torch.nn.functional.silu(f[:, :, 0]) * f[:, :, 1],
            "clamp_glu": (lambda u, v: u * torch.sigmoid(1.702 * u) * (v + 1))(f[:, :, 0].clamp(max=7.0), f[:, :, 1].clamp(-7.0, 7.0))}
    for epi, ref in want.items():
      act = torch.zeros(M, N // 2, dtype=torch.bfloat16, device=gpu)
      C.gemm_wave(xd, ws, act, bd, None, K.EPI[epi], nt, 7.0)
      # one bf16 rounding (2^-9 of the value) behind fp32 arithmetic that differs in its last places
      torch.testing.assert_close(act.cpu().float(), ref.reshape(M, N // 2), rtol=4e-3, atol=1e-3)
  with pytest.raises(RuntimeError):
    C.gemm_wave(xd, ws, torch.zeros(M, N // 2, dtype=torch.bfloat16, device=gpu), None, None, K.EPI["silu"], 1)


@pytest.mark.gpu
@pytest.mark.parametrize("M,H,Hkv,Dh", [(1, 8, 2, 64), (5, 4, 4, 128), (16, 6, 2, 96), (3, 2, 1, 32)])
@pytest.mark.parametrize("bias", [False, True])
def test_rope_and_cache_write(gpu, M, H, Hkv, Dh, bias):
  """q, K and V as the slab reduce with RoPE writes them: rotated in fp32 from the whole sums, padding rows (slot -1) and slots
  past the pool left alone, positions clamped to the table."""
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(Dh + M)
  N, Kd, pages = (H + 2 * Hkv) * Dh, 256, 4
  x, w = integers(g, M, Kd).to(gpu), integers(g, N, Kd).to(gpu)
  b = integers(g, N).to(gpu) if bias else None
  tab = torch.randn(50, Dh, generator=g).to(gpu)
  pos = torch.randint(0, 60, (M,), generator=g, dtype=torch.int32).to(gpu)
  slots = torch.randperm(pages * 64, generator=g)[:M]
  slots[0] = -1 if M > 1 else slots[0]
  slots[-1] = pages * 64 + 3 if M > 4 else slots[-1]
  slots = slots.to(gpu)
  got = []
  for own in (True, False):
    q = torch.zeros(M, H, Dh, dtype=torch.bfloat16, device=gpu)
    kc, vc = torch.zeros(pages, Hkv, 64, Dh, dtype=torch.bfloat16, device=gpu), torch.zeros(pages, Hkv, Dh, 64, dtype=torch.bfloat16, device=gpu)
    if own:
      require().gemm_wave(x, shuffle_for_stream(w), None, b, None, 0, 2, pos=pos, cos_sin=tab, slots=slots, q_out=q, k_cache=kc, v_cache=vc, H=H, Hkv=Hkv)
    else:  # (integer sums: both add up the same numbers)
      require().splitk_rope_kv_write((x.float() @ w.float().t()).contiguous(), 1, b, pos, tab, slots, q, kc, vc, H, Hkv)
    got.append((q, kc, vc))
  for one, other in zip(*got):
    torch.testing.assert_close(one, other, rtol=8e-3, atol=1e-2)  # the last bf16 place (products contracted differently)
    assert torch.equal(one == 0, other == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("D,S", [(128, 1), (2048, 3), (2176, 8), (4096, 4), (8192, 5)])
def test_norm_prologue_is_the_unfused_row(gpu, D, S):
  """One row whose RMS norm runs in the prologue: the residual and the product bit for bit those of the slab
  reduce followed by the plain kernel, with and without the gated epilogue and the rotation."""
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator(device=gpu).manual_seed(D)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  h, lnw, slabs = rn(1, D).to(torch.bfloat16), (1 + 0.1 * rn(D)).to(torch.bfloat16), rn(S, 1, D)
  H, Hkv, Dh = 4, 2, 64
  N = (H + 2 * Hkv) * Dh
  w = shuffle_for_stream((rn(N, D) / D ** 0.5).to(torch.bfloat16))
  w.xot_layout = "stream"
  C, m, xn = require(), h.clone(), torch.empty_like(h)
  C.splitk_resid_rmsnorm(slabs, S, None, m, lnw, xn, 1e-5)  # the sum of the slabs: the row the prologue reads
  p = L.PendingNorm(m.clone(), torch.zeros_like(h), lnw, 1e-5)
  assert torch.equal(L.PendingNorm(m.clone(), torch.zeros_like(h), lnw, 1e-5).materialize(), xn)
  for epi, nt, n in (("none", 1, N), ("none", 4, N), ("silu", 2, N // 2)):
    y, z = (torch.zeros(1, n, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    p.run_wave(w, y, None, epi, nt)
    C.gemm_wave(xn, w, z, None, None, K.EPI[epi], nt)
    assert torch.equal(y, z), (epi, nt)
  assert torch.equal(p.dst, m) and torch.equal(p.src, m)
  tab, pos, slots = rn(16, Dh), torch.tensor([5], dtype=torch.int32, device=gpu), torch.tensor([9], device=gpu)
  got = []
  for fused in (True, False):
    kw = dict(pos=pos, cos_sin=tab, slots=slots, q_out=torch.zeros(1, H, Dh, dtype=torch.bfloat16, device=gpu),
              k_cache=torch.zeros(1, Hkv, 64, Dh, dtype=torch.bfloat16, device=gpu),
              v_cache=torch.zeros(1, Hkv, Dh, 64, dtype=torch.bfloat16, device=gpu), H=H, Hkv=Hkv)
    if fused:
      p.run_wave(w, None, None, "none", 2, **kw)
    else:
      C.gemm_wave(xn, w, None, None, None, 0, 2, **kw)
    got.append([kw[k] for k in ("q_out", "k_cache", "v_cache")])
  assert all(torch.equal(a, b) for a, b in zip(*got))

def test_wave_entries_of_the_tuning_table():
  """A saved choice is taken as it stands; a caller that cannot run the whole-K GEMM passes over its entry; residual products
  keep a table entry of their own where another caller sums the slabs."""
  pol = L.GemmPolicy()
  x, w = torch.zeros(8, 256, dtype=torch.bfloat16), torch.zeros(512, 256, dtype=torch.bfloat16)
  tail = (L._m_bucket(8), 512, 256, "none", False, str(torch.float32))
  cfg = lambda wave, epi="none": pol.shuffled_cfg(x, w, None, None, epi, torch.float32, wave=wave)  # noqa: E731
  pol.table[("sh",) + tail] = ("stream", 1, 4)
  assert cfg("y") == ("stream", 1, 4) and cfg("") == ("stream", 1, 4)
  pol.table[("sh",) + tail] = ("wave", 2, 1)
  pol.table[("shn",) + tail] = ("stream", 2, 1)
  assert cfg("y") == ("wave", 2, 1) and cfg("") == ("stream", 2, 1)
  rtail = (L._m_bucket(8), 512, 256, "resid", False, str(torch.bfloat16))
  pol.table[("sh",) + rtail], pol.table[("shy",) + rtail] = ("stream", 1, 2), ("wave", 1, 1)
  got = [pol.shuffled_cfg(x, w, None, x, "resid", torch.bfloat16, wave=wave) for wave in ("", "y")]
  assert got == [("stream", 1, 2), ("wave", 1, 1)]


def test_wide_candidates_leave_no_cu_idle():
  """17 to 64 rows: widths whose busiest CU has at most 1.4 times an even share of the column tiles, as many tiles as the
  bucket of row counts has row tiles at least (a wave copies at most eight pieces of X), pairs inside a workgroup."""
  cands = lambda *a: [c[1] for c in L.GemmPolicy._wide_cands(*a)]  # noqa: E731
  assert cands(16, 4096, 128, "none", False) == [] == cands(65, 4096, 128, "none", False) == cands(48, 4096, 96, "none", False)
  assert cands(48, 20224, 2048, "none", False) == [5, 6] == cands(33, 20224, 2048, "none", False) and cands(64, 28672, 4096, "silu", False) == [8, 4]
  assert cands(64, 6144, 4096, "none", True) == []
  for M, N, epi, rope in ((17, 256 * 16, "none", False), (64, 28672, "silu", False), (33, 6144, "none", True), (49, 11264, "clamp_glu", False)):
    for nt in cands(M, N, 256, epi, rope):
      assert L._m_bucket(M) // 16 <= nt <= 8 and (nt % 2 == 0 or not (rope or epi in K.GLU_EPI))
      assert -(-(-(-N // 16 // nt)) // 256) * nt * 256 <= 1.4 * (N // 16)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,Kd", [(96, 128), (224, 1408), (128, 2176)])
def test_more_row_tiles_exact(gpu, M, N, Kd):
  """Two to four row tiles on integer operands, bit for bit: a last workgroup with fewer tiles, chunks without a block for every
  wave, a last chunk that is not full, rows past M, every epilogue, rows of a wider buffer; rotation
  and cache write against float64."""
  from xotorch_support_jetson_amd.ops._ext import require
  g = torch.Generator().manual_seed(M + N + Kd)
  x, w, b, r = integers(g, M, Kd), integers(g, N, Kd), integers(g, N), integers(g, M, N)
  full = x.float() @ w.float().t()
  ws, bd, C = shuffle_for_stream(w.to(gpu)), b.to(gpu), require()
  wide = torch.zeros(M, Kd + 16, dtype=torch.bfloat16, device=gpu)
  wide[:, 8:8 + Kd] = x.to(gpu)
  xd = wide[:, 8:8 + Kd]
  f = (full + b.float()).view(M, N // 32, 2, 16)
  want = {"silu": torch.nn.functional.silu(f[:, :, 0]) * f[:, :, 1],
          "clamp_glu": (lambda u, v: u * torch.sigmoid(1.702 * u) * (v + 1))(f[:, :, 0].clamp(max=7.0), f[:, :, 1].clamp(-7.0, 7.0))}
  for nt in range(1, 9):
    y = torch.full((M + 1, N), 5.0, device=gpu)
    if nt < -(-M // 16):
      with pytest.raises(RuntimeError):
        C.gemm_wave(xd, ws, y[:M], bd, None, K.EPI["none"], nt)
      continue
    C.gemm_wave(xd, ws, y[:M], bd, None, K.EPI["none"], nt)
    assert torch.equal(y[:M].cpu(), full + b.float()) and bool((y[M] == 5.0).all()), nt
    h = r.to(gpu)
    C.gemm_wave(xd, ws, h, None, h, K.EPI["resid"], nt)
    assert torch.equal(h.cpu(), (full + r.float()).to(torch.bfloat16)), nt
    a = torch.zeros(M, N, dtype=torch.bfloat16, device=gpu)
    C.gemm_wave(xd, ws, a, None, None, K.EPI["relu2"], nt)
    assert torch.equal(a.cpu(), full.clamp(min=0).square().to(torch.bfloat16)), nt
    for epi, ref in want.items():
      act = torch.zeros(M, N // 2, dtype=torch.bfloat16, device=gpu)
      if nt % 2:
        with pytest.raises(RuntimeError):
          C.gemm_wave(xd, ws, act, bd, None, K.EPI[epi], nt, 7.0)
        continue
      C.gemm_wave(xd, ws, act, bd, None, K.EPI[epi], nt, 7.0)
      # one bf16 rounding (2^-9 of the value) behind fp32 arithmetic that differs in its last places
      torch.testing.assert_close(act.cpu().float(), ref.reshape(M, N // 2), rtol=4e-3, atol=1e-3)
  H, Hkv, Dh, pages = N // 32 - 2, 1, 32, 2
  tab = torch.randn(70, Dh, generator=g)
  c, sn = tab[:M, None, :16].double(), tab[:M, None, 16:].double()
  lo, hi = (t.double() for t in full.view(M, H + 2, 2, 16).unbind(2))
  rot = torch.cat([lo * c - hi * sn, hi * c + lo * sn], -1)
  slots = torch.randperm(pages * 64, generator=g)[:M]
  slots[M // 2] = -1
  live = slots >= 0
  for nt in (n for n in (2, 4, 6, 8) if n >= -(-M // 16)):
    q = torch.zeros(M, H, Dh, dtype=torch.bfloat16, device=gpu)
    kc, vc = torch.zeros(pages, Hkv, 64, Dh, dtype=torch.bfloat16, device=gpu), torch.zeros(pages, Hkv, Dh, 64, dtype=torch.bfloat16, device=gpu)
    C.gemm_wave(xd, ws, None, None, None, 0, nt, pos=torch.arange(M, dtype=torch.int32, device=gpu), cos_sin=tab.to(gpu),
                slots=slots.to(gpu), q_out=q, k_cache=kc, v_cache=vc, H=H, Hkv=Hkv)
    # one bf16 rounding of two products of whole numbers (below 2^14, so exact to 2^-10 in fp32)
    torch.testing.assert_close(q.cpu().double(), rot[:, :H], rtol=4e-3, atol=2e-3)
    torch.testing.assert_close(kc.cpu().double().view(-1, Dh)[slots[live]], rot[live, H], rtol=4e-3, atol=2e-3)
    # (a page of V: 8 chunks of 8 keys, [Dh][8] each)
    values = vc.cpu().view(pages, 8, Dh, 8).transpose(2, 3).reshape(-1, Dh)
    assert torch.equal(values[slots[live]], full.view(M, H + 2, Dh)[live, H + 1].to(torch.bfloat16))
    untouched = torch.ones(pages * 64, dtype=torch.bool).index_fill_(0, slots[live], False)
    assert not kc.cpu().view(-1, Dh)[untouched].any() and not values[untouched].any()


def test_loads_past_an_operand_are_bounds_checked():
  """A buffer load's scalar offset is no part of its bounds check, so a load that may pass the end of its operand (a chunk past K,
  a stage past the last one) carries its place in the vector offset.  The exceptions are named: `inside` is within the operand
  for all lanes, and loads to LDS go stage by stage through whole tiles."""
  csrc = pathlib.Path(L.__file__).parents[1] / "csrc"
  calls = [(f.name, a) for f in sorted(csrc.glob("*.hip")) for a in re.findall(r"amdgcn_raw_buffer_load_b\d+\(([^()]*(?:\([^()]*\)[^()]*)*)\)", f.read_text())]
  assert {"gemm_wave.hip", "gemm_group.hip", "recurrence_chunk.hip"} <= {f for f, _ in calls}
  assert not [(f, a) for f, a in calls if a.split(",")[-2].strip() not in ("0", "inside")]
  group = (csrc / "gemm_group.hip").read_text()  # its weights: the slice's last block at most
  assert re.findall(r"buf16nt\(wr,.*\)", group) == ["buf16nt(wr, lane * 16, min(ch * U + u, nb - 1) * 1024)"]
