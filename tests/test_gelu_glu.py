"""gelu_tanh(gate) * up in the epilogue of the dense projections, every kernel configuration the policy would try."""
import pytest
import torch

from xotorch_support_jetson_amd.models.weights import interleave_gate_up

F64 = torch.float64


def want_of(x, g, u):
  z = x.double() @ g.double().T
  gelu = 0.5 * z * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (z + 0.044715 * z ** 3)))
  return gelu * (x.double() @ u.double().T), z


@pytest.mark.gpu
@pytest.mark.parametrize("M", [65, 130, 520, 1024, 2100])
@pytest.mark.parametrize("N,D", [(256, 128), (512, 384), (768, 1024)])
def test_gelu_glu_epilogue(M, N, D):
  from xotorch_support_jetson_amd.ops import linear as L
  gen = torch.Generator().manual_seed(M + N)
  x = torch.randn(M, D, generator=gen).bfloat16()
  w = (torch.randn(N, D, generator=gen) * (3 * D ** -0.5)).bfloat16()  # gates of +-10: both tails of the tanh
  want, z = want_of(x, w[:N // 2], w[N // 2:])
  xd, ws = x.cuda(), L.to_stream_layout(interleave_gate_up(w[:N // 2], w[N // 2:]).contiguous().cuda())
  cands = [c for c in L.policy._big_cands(M, N, D) if c[1] in (2256, 128, 4256)]
  assert cands
  for cfg in cands + ["as chosen"]:
    out = torch.full((M, N // 2), 7.0, dtype=torch.bfloat16, device="cuda")
    if cfg == "as chosen":
      L.linear(xd, ws, epi="gelu_glu", out=out)
    else:
      L._shuffled_call(xd, ws, None, None, "gelu_glu", out, cfg)
    # half a bf16 step of the result, and the fp32 sums' error (products of magnitude |x||w|, sqrt(D) of them at random
    # signs, so within 2^-24 D of the operands' scale) through the gate's slope (at most 1.13) and the other factor
    err = (out.double().cpu() - want).abs()
    lim = want.abs() * 2.0 ** -8 + 2.0 ** -24 * D * 9 * (1 + z.abs()) * 4
    assert bool((err <= lim).all()), (cfg, float((err / lim).max()))


@pytest.mark.gpu
def test_gelu_glu_epilogue_extremes():
  """Huge gates give the activation's limits, zero gates (the padding rows) 0."""
  from xotorch_support_jetson_amd.ops import linear as L
  vals = [0.0, -0.0, 3e38, -3e38]
  for M in (65, 300):
    x = torch.zeros(M, 128, dtype=torch.bfloat16)
    w = torch.zeros(256, 128, dtype=torch.bfloat16)
    w[:128, 0] = 1.0
    w[128:, 1] = 1.0
    x[:, 1] = 2.0
    for i in range(M):
      x[i, 0] = vals[i % 4]
    ws = L.to_stream_layout(interleave_gate_up(w[:128], w[128:]).contiguous().cuda())
    out = L.linear(x.cuda(), ws, epi="gelu_glu").float().cpu()
    for i in range(M):
      v = vals[i % 4]
      # (0 * anything stays 0 in the sums: 3e38 and 2 are the only terms of their columns; 6e38 overflows to infinity)
      assert bool((out[i] == (float("inf") if v > 1e38 else 0.0)).all()), (M, v, out[i, :2])


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("T,F,off,pad", [(1, 16, 0, 0), (5, 40, 12, 0), (7, 100, 64, 28), (3, 33, 5, 3)])
def test_gelu_mul_of_tiles(dev, T, F, off, pad):
  """Gate and up columns in alternating tiles of 16, whole vectors or not, against the two-run form (bit for bit)."""
  from xotorch_support_jetson_amd.ops import kernels as K
  n = -(-F // 16) * 16
  gu = torch.randn(T, 2, n, generator=torch.Generator().manual_seed(F))
  P = torch.zeros(T, off + 2 * n + pad)
  P[:, off:off + 2 * n] = gu.reshape(T, 2, n // 16, 16).transpose(1, 2).reshape(T, 2 * n)
  for dt in (torch.float32, torch.bfloat16):
    got, want = (torch.zeros(T, n + 4, dtype=dt, device=dev) for _ in range(2))
    K.gelu_mul(P.to(dev), off, -1, F, got)
    K.gelu_mul(gu.reshape(T, 2 * n).to(dev), 0, n, F, want)
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_gelu_mul_refuses_columns_outside_the_projection():
  from xotorch_support_jetson_amd.ops import kernels as K
  P, out = torch.zeros(2, 64, device="cuda"), torch.zeros(2, 16, device="cuda")
  for gate, up in ((0, -2), (0, -16), (-1, 16), (0, 49), (33, -1)):
    with pytest.raises(RuntimeError):
      K.gelu_mul(P, gate, up, 16, out)
  K.gelu_mul(P, 32, -1, 16, out)


@pytest.mark.gpu
@pytest.mark.parametrize("ff", [192, 130, 640])
@pytest.mark.parametrize("T", [65, 300, 1030])
def test_parallel_block_in_two_products(ff, T, monkeypatch):
  """The gate / up rows at the end of a parallel block's fused projection in a GEMM of their own (long steps), and one GEMM with
  the pass over its result, against float64: the other columns, the activation, its zero K padding."""
  import types

  from xotorch_support_jetson_amd.models import config, transformer, weights
  from xotorch_support_jetson_amd.ops import linear as L
  c = config.from_hf_config(dict(config.TINY_TAREPEL, layers=[dict(config.TINY_TAREPEL["layers"][0], mlp={"kind": "dense", "ff": ff})]))
  get = {k: v.bfloat16().float() for k, v in weights.random_mixed_tensors(c, ff).items()}.__getitem__
  lw = weights.build_mixed_layer(c.layer_specs[0], get, "l0.", 128, "cuda", torch.bfloat16)
  lw.in_w = L.to_stream_layout(lw.in_w)
  assert L.layout_of(lw.in_w) == "stream"
  x = torch.randn(T, 128, generator=torch.Generator().manual_seed(T)).bfloat16()
  epis, real = [], transformer.linear
  monkeypatch.setattr(transformer, "linear", lambda *a, **k: (epis.append(k.get("epi")), real(*a, **k))[1])
  z, u = (x.double() @ get(f"l0.mlp.{n}").double().T for n in ("gate", "up"))
  want = 0.5 * z * (1 + torch.tanh(0.7978845608028654 * (z + 0.044715 * z ** 3))) * u
  for split in (True, False):
    monkeypatch.setattr(transformer, "GELU_EPI_ROWS", 1 if split else T + 1)
    monkeypatch.setattr(transformer, "GELU_EPI_SIZE", 1)
    P, act = transformer.ShardModel._in_and_act(
      types.SimpleNamespace(_proj=transformer.ShardModel._proj), x.cuda(), lw,
      lambda name, live, padded: torch.zeros(T, padded, dtype=torch.bfloat16, device="cuda"))
    P, act = P.cpu().double(), act.cpu().double()
    assert epis.count("gelu_glu") == 1
    assert act.shape[1] == lw.down_w.shape[1] >= ff and bool((act[:, ff:] == 0).all())
    # half a bf16 step (2^-9) of the value, and fp32 sums of 128 products in front of it
    assert bool(((act[:, :ff] - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max()).all())
    for name, w in weights.mixed_layer_names(c.layer_specs[0], "l0.")["in"]:
      (o, n), ref = lw.cols[name], x.double() @ get(w).double().T
      assert o + n <= lw.cols["gate_up"][0] and bool(((P[:, o:o + n] - ref).abs() <= 1e-5 * ref.abs().max()).all())
