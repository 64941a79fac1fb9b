"""Host-side dispatch policy (CPU): decode-attention partitioning per batch / block-table width, and the
GEMM tuner's split-K slab charge.  The kernels these choices select are covered in tests/test_kernels_gpu.py."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L


def test_decode_partition_defaults():
  ws = K.DecodeWorkspace(512, 64, 128, 8192, torch.device("cpu"), algo=-1)
  # few (sequence, KV head) pairs: 4-wave workgroups over 4-page partitions, merged by the reduce launch
  assert ws.partition(1, 8, 32) == (4, 8, 0)
  # many pairs: the waves of a workgroup share a unit
  ppp, nparts, algo = ws.partition(512, 8, 9)
  assert algo == 3 and ppp * nparts >= 9  # non-temporal page loads



def test_decode_partition_small_batch():
  ws = K.DecodeWorkspace(8, 32, 128, 4096, torch.device("cpu"), algo=-1)
  assert ws.partition(1, 8, 16)[2] == 0 and ws.partition(1, 8, 32)[2] == 0  # the workgroup kernel, split
  assert ws.partition(8, 8, 8)[2] == 2  # 64 pairs: shared units (cache-resident pages: plain loads)
  assert K.DecodeWorkspace(64, 32, 128, 8192, torch.device("cpu"), algo=-1).partition(64, 8, 128)[2] == 3  # 2 GB: nt
  fixed = K.DecodeWorkspace(8, 32, 128, 4096, torch.device("cpu"), pages_per_part=4, algo=-1)
  assert fixed.partition(1, 8, 16)[2] == 0  # an explicit partition size is honoured


def test_slab_charge(monkeypatch):
  assert L._slab_read_ms(("big", 256, 1), 512, 8192) == 0.0
  four = L._slab_read_ms(("big", 256, 4), 512, 8192)
  assert abs(four - 4 * 512 * 8192 * 4 / (L.SLAB_TBPS * 1e9)) < 1e-12
  assert L._slab_read_ms(("big", 256, 2), 512, 8192) * 2 == four
  monkeypatch.setattr(L, "SLAB_TBPS", 0.0)
  assert L._slab_read_ms(("big", 256, 4), 512, 8192) == 0.0


def test_tuner_tie_break_prefers_ping_pong(monkeypatch):
  """Within XOT_GEMM_TIE of the fastest, a 256-row tile variant at the same K split gives way to the ping-pong
  256 x 256 tile; other kernels and other splits keep the plain minimum."""
  t = {("big", 224, 1): 0.400, ("big", 1256, 1): 0.408, ("big", 256, 1): 0.401, ("big", 1256, 2): 0.399}
  assert L._tie_break(t) == ("big", 1256, 2)  # the fastest is already a ping-pong config
  t.pop(("big", 1256, 2))
  assert L._tie_break(t) == ("big", 1256, 1)
  t[("big", 1256, 1)] = 0.500  # beyond the tie window: the next preference inside it
  assert L._tie_break(t) == ("big", 256, 1)
  assert L._tie_break({("stream", 2, 4): 0.1, ("big", 1256, 1): 0.101}) == ("stream", 2, 4)
  monkeypatch.setattr(L, "TIE", 0.0)
  assert L._tie_break({("big", 224, 1): 0.4, ("big", 1256, 1): 0.401}) == ("big", 224, 1)


def test_tuner_offers_two_phase_ping_pong(monkeypatch):
  """The two-phase ping-pong tile (2256) is a gemm_big candidate and the first choice inside the tie window."""
  codes = {c[1] for c in L.GemmPolicy._big_cands(512, 57344, 8192)}
  assert {256, 1256, 2256, 128} <= codes
  assert L._tie_break({("big", 1256, 1): 0.40, ("big", 2256, 1): 0.41}) == ("big", 2256, 1)
  # across K splits only the two-phase tile gets a (wider) window
  t = {("big", 128, 2): 0.843, ("big", 2256, 4): 0.927, ("big", 256, 4): 0.90}
  assert L._tie_break(t) == ("big", 2256, 4)
  t[("big", 2256, 4)] = 0.95
  assert L._tie_break(t) == ("big", 128, 2)
  # short row tiles: the two-phase 192-row tile is offered and preferred like the 256-row one
  assert ("big", 1922256, 1) in L.GemmPolicy._big_cands(384, 8192, 8192)
  assert L._tie_break({("big", 1920256, 2): 0.50, ("big", 1922256, 2): 0.51}) == ("big", 1922256, 2)
  t = {("big", 128, 4): 55.0, ("big", 2256, 6): 59.6}  # across K splits half of that between 512 and the tall rows
  assert [L._tie_break(t, M)[1] for M in (512, 513, 911, L.W4_PREF_M - 1)] == [2256, 128, 128, 128]
  monkeypatch.setattr(L, "TIE_X", 0.0)
  assert L._tie_break({("big", 128, 2): 0.843, ("big", 2256, 4): 0.85}) == ("big", 128, 2)
  monkeypatch.setattr(L, "PP2", False)
  assert 2256 not in {c[1] for c in L.GemmPolicy._big_cands(512, 57344, 8192)}


def test_cpu_reference_linear_caches_fp32_weights():
  """The CPU path widens a low-precision weight once and reuses it, re-widening after an in-place write (a
  trained weight written back) and never caching a weight that requires grad."""
  from xotorch_support_jetson_amd.ops import reference as ref
  torch.manual_seed(0)
  x = torch.randn(3, 64)
  w = torch.randn(32, 64).to(torch.bfloat16)
  y1 = ref.linear(x, w)
  assert hasattr(w, "_xot_f32")
  f32 = w._xot_f32[1]
  assert ref.linear(x, w) is not None and w._xot_f32[1] is f32  # reused
  w.mul_(2)
  y2 = ref.linear(x, w)
  assert torch.allclose(y2, 2 * y1, rtol=1e-2, atol=1e-2)
  wg = torch.randn(32, 64, requires_grad=True)
  ref.linear(x, wg.to(torch.bfloat16))
  assert not hasattr(wg, "_xot_f32")


def test_tuner_prefers_four_wave_tile_on_tall_gemms(monkeypatch):
  """The four-wave 256 x 256 tile (4256) is a candidate wherever N % 256 == 0; from W4_PREF_M rows it takes the
  ping-pong tile's place as first choice inside the tie windows, below it the ping-pong tile keeps it."""
  assert 4256 in {c[1] for c in L.GemmPolicy._big_cands(4096, 4096, 4096)}
  assert 4256 not in {c[1] for c in L.GemmPolicy._big_cands(4096, 4096 + 224, 4096)}
  t = {("big", 2256, 1): 0.40, ("big", 4256, 1): 0.41}
  assert L._tie_break(t, 4096) == ("big", 4256, 1)
  assert L._tie_break(t, 512) == ("big", 2256, 1)
  t = {("big", 2256, 2): 0.40, ("big", 4256, 1): 0.43}  # across K splits: the preferred tile's wider window
  assert L._tie_break(t, 4096) == ("big", 4256, 1)
  monkeypatch.setattr(L, "W4", False)
  assert 4256 not in {c[1] for c in L.GemmPolicy._big_cands(4096, 4096, 4096)}


def test_tall_gemms_take_the_four_wave_tile_untimed(monkeypatch):
  """M >= W4_PREF_M: ('big', 4256, 1) straight away (no cold-timing pass inside the first prefill chunk; two K halves of a
  long K: below), except a
  residual epilogue into fp32 (the tile has none); XOT_GEMM_TALL_TUNE=1 times them again."""
  pol = L.GemmPolicy()
  x, w = torch.empty(4096, 1024, dtype=torch.bfloat16), torch.empty(2048, 1024, dtype=torch.bfloat16)
  assert pol.shuffled_cfg(x, w, None, None, "none", torch.bfloat16) == ("big", 4256, 1)
  assert pol.shuffled_cfg(x, w, None, None, "none", torch.float32) == ("big", 4256, 1)
  monkeypatch.setattr(L, "TALL_FIXED", False)
  monkeypatch.setattr(L.GemmPolicy, "_no_tuning", lambda self: True)  # the heuristic instead of a GPU timing
  pol2 = L.GemmPolicy()
  assert pol2.shuffled_cfg(x, w, None, None, "none", torch.bfloat16)[0] == "big"


def test_tall_k_halves_follow_the_rows_of_the_call(monkeypatch):
  """Two K halves where 256-row tiles fill at most half the CUs, whatever M of the bucket came before: from K 8192 for residual
  products, from 24576 for plain ones."""
  monkeypatch.setattr(L.GemmPolicy, "_no_tuning", lambda self: False)
  sized = []
  monkeypatch.setattr(L.scratch, "splitk", lambda dev, n, slot=0: sized.append(n))

  def splits(pol, M, N, Kd, epi="none"):
    x, w = torch.empty(M, Kd, dtype=torch.bfloat16, device="meta"), torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")
    kind, code, S = pol.shuffled_cfg(x, w, None, None, epi, torch.bfloat16)
    assert (kind, code) == ("big", 4256)
    return S
  for N, last in ((4096, 2048), (5120, 1536), (6144, 1280)):
    for Ms in ((1100, 2048), (2048, 1100)):
      pol = L.GemmPolicy()
      for M in Ms:
        half = M <= last
        assert splits(pol, M, N, 14336, "resid") == (2 if half else 1)
        assert splits(pol, M, N, 14336) == 1
        for epi in ("none", "resid"):
          assert splits(pol, M, N, 24576, epi) == (2 if half else 1)
        assert splits(pol, M, N, 4096, "resid") == 1
      assert not any(k[0].startswith("sh") and k[1] == 2048 and k[2] == N for k in pol.table)
  assert sized and max(sized) == 2 * 2048 * 4096
  monkeypatch.setattr(L.GemmPolicy, "_no_tuning", lambda self: True)  # under capture: nothing to size
  assert splits(L.GemmPolicy(), 2048, 4096, 28672) == 1


@pytest.mark.parametrize("M,N,Kd,parts", [(1024, 2048, 2048, 3), (1280, 2048, 5632, 3), (1281, 2048, 5632, 2), (1663, 2048, 4096, 2),
                                          (2048, 2048, 2048, 2), (2049, 2048, 2048, 1), (1663, 2048, 1920, 1), (4096, 1024, 2048, 2),
                                          (1024, 4096, 2048, 2), (1025, 4096, 2048, 1), (1664, 2048, 24576, 2)])
def test_tall_parts_that_the_next_pass_sums(monkeypatch, M, N, Kd, parts):
  """A product whose slabs the pass behind it sums is cut where 128-row tiles fill at most half the CUs, into no more than one round."""
  monkeypatch.setattr(L.GemmPolicy, "_no_tuning", lambda self: False)
  sized = []
  monkeypatch.setattr(L.scratch, "splitk", lambda dev, n, slot=0: sized.append(n))
  x, w = (torch.empty(r, Kd, dtype=torch.bfloat16, device="meta") for r in (M, N))
  for epi, dt in (("none", torch.float32), ("resid", torch.bfloat16)):
    assert L.GemmPolicy().shuffled_cfg(x, w, None, None, epi, dt, summed=True) == ("big", 4256, parts)
    whole = L.GemmPolicy().shuffled_cfg(x, w, None, None, epi, dt)
    assert whole == ("big", 4256, 2 if Kd == 24576 else 1)
  assert sized == ([parts * M * N] * len(sized)) and (parts == 1) == (not sized)
  monkeypatch.setattr(L.GemmPolicy, "_no_tuning", lambda self: True)
  assert L.GemmPolicy().shuffled_cfg(x, w, None, None, "none", torch.float32, summed=True) == ("big", 4256, 1)


def test_qkv_projection_is_timed_with_what_follows_it(monkeypatch):
  """linear_rope_kv's choice: the rotation and the KV write behind a whole product, one launch behind slabs, are part of the time, so
  a whole product that is the faster one by itself does not win."""
  M, H, Hkv, Dh, D = 300, 4, 2, 64, 512
  N, ran = (H + 2 * Hkv) * Dh, []
  x, w = (torch.empty(*s, dtype=torch.bfloat16, device="meta") for s in ((M, D), (N, D)))
  kc, vc = torch.empty(8, Hkv, 64, Dh, dtype=torch.bfloat16, device="meta"), torch.empty(8, Hkv, Dh, 64, dtype=torch.bfloat16, device="meta")
  took = {"whole": 10.0, "slabs": 10.1, "write": 9.0, "rotate": 9.0 - 5.0}
  clock = [0.0]

  def step(name, got=None):
    return lambda *a, **k: (ran.append(name), clock.__setitem__(0, clock[0] + took[name]), got)[2]

  def timed(fn):
    clock[0] = 0.0
    fn()
    return clock[0]

  class Lib:
    splitk_rope_kv_write = staticmethod(step("rotate"))
  pol = L.GemmPolicy()
  pol._path_resolved = True
  for name, value in (("_no_tuning", lambda self: False), ("_time", staticmethod(timed)),
                      ("_big_cands", staticmethod(lambda *a: [("big", 128, 1), ("big", 128, 2)])), ("_stream_cands", staticmethod(lambda *a: []))):
    monkeypatch.setattr(L.GemmPolicy, name, value)
  monkeypatch.setattr(L, "policy", pol)
  monkeypatch.setattr(L.scratch, "splitk", lambda dev, n, slot=0: torch.empty(n, device="meta"))
  monkeypatch.setattr(L, "_shuffled_call", step("whole"))
  monkeypatch.setattr(L, "_slab_call", step("slabs"))
  monkeypatch.setattr(L.K, "rope_kv_write", step("write"))
  monkeypatch.setattr(L, "require", lambda: Lib)
  monkeypatch.setattr(L, "layout_of", lambda w: "stream")
  monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
  L.linear_rope_kv(x, w, None, None, None, None, kc, vc, H, Hkv)
  assert list(pol.table.values()) == [("big", 128, 2)] and ran[-2:] == ["slabs", "rotate"] and ran.count("whole") == ran.count("write") == 1


@pytest.mark.parametrize("whole", [True, False])
def test_a_timed_run_is_not_charged_for_its_slabs_again(monkeypatch, whole):
  """Where the caller's whole step is timed, the read of the slabs lies in the timing; a product alone is charged for it."""
  M, N, Kd = 512, 3072, 2048
  read = L._slab_read_ms(("big", 128, 4), M, N)
  took = {("big", 128, 1): 1.0, ("big", 128, 4): 1.0 - read / 2}
  pol, now = L.GemmPolicy(), []
  pol._path_resolved = True
  for name, value in (("_no_tuning", lambda self: False), ("_time", staticmethod(lambda fn: (fn(), took[now[-1]])[1])),
                      ("_big_cands", staticmethod(lambda *a: list(took))), ("_stream_cands", staticmethod(lambda *a: []))):
    monkeypatch.setattr(L.GemmPolicy, name, value)
  monkeypatch.setattr(L, "_shuffled_call", lambda x, w, b, r, e, y, cfg: now.append(cfg))
  monkeypatch.setattr(L.scratch, "splitk", lambda dev, n, slot=0: None)
  x, w = (torch.empty(*s, dtype=torch.bfloat16, device="meta") for s in ((M, Kd), (N, Kd)))
  got = pol.shuffled_cfg(x, w, None, None, "none", torch.bfloat16, run=now.append if whole else None)
  assert got == ("big", 128, 4 if whole else 1)


def test_untuned_choice_without_stream_candidates(monkeypatch):
  """The GELU pair epilogue is built for the tall tiles alone: a choice without a timing pass takes one of them at any row count."""
  monkeypatch.setattr(L.GemmPolicy, "_no_tuning", lambda self: True)
  w = torch.empty(512, 256, dtype=torch.bfloat16)
  for M in (L.BIG_MIN_M, 100, 128, 129, 700):
    x = torch.empty(M, 256, dtype=torch.bfloat16)
    got = L.GemmPolicy().shuffled_cfg(x, w, None, None, "gelu_glu", torch.bfloat16)
    assert got[0] == "big" and got[1] in (2256, 128, 4256)
    assert L.GemmPolicy().shuffled_cfg(x, w, None, None, "none", torch.bfloat16)[0] == ("stream" if M <= 128 else "big")


def test_seed_table_parses_and_loads_under_the_box_table(tmp_path):
  """ops/gemm_seed_mi355x.json: comment keys skipped, the headline decode picks load, and a key the box tuned itself
  keeps the box's choice (the seed only fills gaps)."""
  import json
  from xotorch_support_jetson_amd.ops import linear as L
  pol = L.GemmPolicy()
  own = ("sh", 512, 10240, 8192, "none", False, "torch.bfloat16")
  pol.table[own] = ("big", 256, 2)  # as if the box had tuned it
  pol._load(L.SEED_TABLE)
  assert pol.table[own] == ("big", 256, 2)
  assert pol.table[("sh", 512, 57344, 8192, "silu", False, "torch.bfloat16")] == ("big", 2256, 1)
  assert not any(isinstance(k, tuple) and k and str(k[0]).startswith("_") for k in pol.table)
  assert all(k.startswith("_") or json.loads(k)[0] == "sh" for k in json.load(open(L.SEED_TABLE)))
