"""Whole-K decode GEMM of single column tiles (csrc/gemm_wave.hip gemm_solo_kernel): row counts at the edges of its LDS rows, K that
leaves waves without blocks, both column splits, residual and bias, against float32."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops import linear as L


def test_shapes_it_takes():
  assert L.solo_fits(1, 2048, 8192) and L.solo_fits(8, 4096, 128)
  assert not (L.solo_fits(9, 2048, 8192) or L.solo_fits(1, 4112, 8192) or L.solo_fits(1, 2048, 8192 + 64) or L.solo_fits(1, 2056, 8192))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,Kd", [(64, 128), (2048, 2048), (2048, 2816), (192, 5632), (2112, 4224), (4096, 8192)])
def test_solo(M, N, Kd):
  g = torch.Generator(device="cuda").manual_seed(M * N + Kd)
  big = torch.randn(M + 1, Kd + 8, generator=g, device="cuda").bfloat16()
  big[:, Kd:] = float("inf")  # (behind the rows: never a factor)
  big[M] = float("nan")
  x = big[:M, :Kd]
  w = (torch.randn(N, Kd, generator=g, device="cuda") * Kd ** -0.5).bfloat16()
  ws = L.to_stream_layout(w)
  bias = torch.randn(N, generator=g, device="cuda").bfloat16()
  want = x.float() @ w.float().t()
  C = K.require()
  y = torch.empty(M, N, device="cuda")
  if M > L.SOLO_MAX_M:
    with pytest.raises(RuntimeError):
      C.gemm_wave(x, ws, y, None, None, 0, 0)
    return
  C.gemm_wave(x, ws, y, None, None, 0, 0)
  # fp32 sums of bf16 products in another order: Kd terms of about Kd ** -0.5, rounding 2^-24 of partial sums of a few units
  assert float((y - want).abs().max()) < 1e-5 * Kd ** 0.5
  C.gemm_wave(x, ws, y, bias, None, 0, 0)
  assert float((y - (want + bias.float())).abs().max()) < 1e-5 * Kd ** 0.5
  h = torch.randn(M, N, generator=g, device="cuda").bfloat16()
  full = want + bias.float() + h.float()
  C.gemm_wave(x, ws, h, bias, h, 1, 0)  # in place
  assert bool(((h.float() - full).abs() <= 2.0 ** -8 * full.abs() + 1e-5 * Kd ** 0.5).all())  # one rounding to bf16


@pytest.mark.gpu
@pytest.mark.parametrize("epi", [2, 3, 4])
def test_solo_refuses_other_epilogues(epi):
  w = L.to_stream_layout(torch.zeros(64, 128, device="cuda", dtype=torch.bfloat16))
  x, y = torch.zeros(1, 128, device="cuda", dtype=torch.bfloat16), torch.zeros(1, 64 if epi == 4 else 32, device="cuda", dtype=torch.bfloat16)
  with pytest.raises(RuntimeError):
    K.require().gemm_wave(x, w, y, None, None, epi, 0)


@pytest.mark.gpu
def test_pending_norm_without_slabs():
  """One row: the projection sums by itself and the next product's prologue norms its row; materialize() leaves the same."""
  g = torch.Generator(device="cuda").manual_seed(5)
  x, h = (torch.randn(1, n, generator=g, device="cuda").bfloat16() for n in (5632, 2048))
  w = L.to_stream_layout((torch.randn(2048, 5632, generator=g, device="cuda") * 0.02).bfloat16())
  ln = torch.rand(2048, generator=g, device="cuda").bfloat16()
  h2, other = h.clone(), torch.zeros_like(h)
  p = L.linear_resid_norm(x, w, h2, ln, 1e-5, defer_to=other)
  assert isinstance(p, L.PendingNorm)
  ref = (x.float() @ L.to_rowmajor(w).float().t() + h.float())
  want = K.rmsnorm(h2, ln, 1e-5)[0]
  assert float((h2.float() - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max()) + 1e-3
  assert torch.equal(p.materialize(), want) and torch.equal(other, h2)
  other.zero_()
  wn = L.to_stream_layout((torch.randn(4096, 2048, generator=g, device="cuda") * 0.02).bfloat16())
  got = L.linear(L.linear_resid_norm(x, w, h.clone(), ln, 1e-5, defer_to=other), wn)
  assert torch.equal(other, h2)
  assert float((got.float() - want.float() @ L.to_rowmajor(wn).float().t()).abs().max()) < 2e-2 * float(got.float().abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hkv,Dh,N", [(32, 8, 64, 2048), (32, 8, 128, 4096), (14, 2, 64, 896), (1, 1, 128, 64)])
def test_merge_of_a_lone_sequence(H, Hkv, Dh, N):
  """Parts merged in the output projection's prologue, bit for bit the attention's own merge and the product of its row."""
  width, Kd = 16, H * Dh
  g = torch.Generator(device="cuda").manual_seed(H)
  kc = torch.randn(width, Hkv, 64, Dh, generator=g, device="cuda").bfloat16()
  vc = torch.randn(width, Hkv, Dh, 64, generator=g, device="cuda").bfloat16()
  bt = torch.randperm(width, generator=g, device="cuda").int()[None].contiguous()
  q = torch.randn(1, H, Dh, generator=g, device="cuda").bfloat16()
  w = L.to_stream_layout((torch.randn(N, Kd, generator=g, device="cuda") * 0.02).bfloat16())
  bias, h0 = torch.randn(N, generator=g, device="cuda").bfloat16(), torch.randn(1, N, generator=g, device="cuda").bfloat16()
  ws = K.DecodeWorkspace(1, H, Dh, width * 64, q.device)
  ln = torch.ones(N, device="cuda", dtype=torch.bfloat16)
  assert L.merge_fits(w)
  for n in (0, 1, 256, 257, 600, width * 64):
    cl = torch.tensor([n], dtype=torch.int32, device="cuda")
    a = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws, plan=K.LONE)
    h1, h2 = h0.clone(), h0.clone()
    y1 = L.linear_resid_norm(a.view(1, Kd), w, h1, ln, 1e-5, bias=bias)
    p = K.attn_decode(q, kc, vc, bt, cl, Dh ** -0.5, ws, defer_merge=True, plan=K.LONE)
    assert isinstance(p, K.PendingMerge)
    assert torch.equal(L.linear_resid_norm(p, w, h2, ln, 1e-5, bias=bias), y1) and torch.equal(h1, h2), n
