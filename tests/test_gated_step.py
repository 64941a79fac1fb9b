"""Chunk-local sigmoid attention of single tokens (csrc/mixers.hip attn_gated_step_k): page and chunk edges, waves without a page, every
group size it takes, empty rows, slots that no token has written, against float64; fp32 weights keep their precision."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K


def _exact(q, kc, vc, bt, lens, pb, scale, chunk, out_scale):
  T, H, d = q.shape
  G = kc.shape[1]
  out = torch.zeros(T, H, d, dtype=torch.float64, device=q.device)
  for t, n in enumerate(lens):
    if n == 0:
      continue
    pos = n - 1
    lo = pos // chunk * chunk
    pages = bt[t, :pos // 64 + 1].long()
    k = kc[pages].double().transpose(1, 2).reshape(-1, G, d)[lo:n]
    v = vc[pages].double().permute(0, 3, 1, 2).reshape(-1, G, d)[lo:n]
    k, v = (x.repeat_interleave(H // G, 1) for x in (k, v))
    w = torch.sigmoid(torch.einsum("hd,khd->kh", q[t].double(), k) * scale + pb.double())
    out[t] = torch.einsum("kh,khd->hd", w, v) * out_scale
  return out.reshape(T, H * d)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,d", [(16, 4, 128), (16, 1, 64), (6, 6, 96), (32, 4, 32), (12, 1, 128)])
@pytest.mark.parametrize("chunk", [1024, 96, 64, 7])
@pytest.mark.parametrize("rep", [1, 30])
def test_gated_step(H, G, d, chunk, rep):
  g = torch.Generator(device="cuda").manual_seed(H + d + chunk)
  lens = [1, 7, 63, 64, 65, 96, 97, 128, 129, 300, 0, 600] * rep
  T, width = len(lens), 10
  pages = sum(-(-n // 64) for n in lens) + 1
  kc = torch.randn(pages, G, 64, d, generator=g, device="cuda").bfloat16()
  vc = torch.randn(pages, G, d, 64, generator=g, device="cuda").bfloat16()
  perm, at = torch.randperm(pages, generator=g, device="cuda").int().cpu(), 0
  bt = torch.zeros(T, width, dtype=torch.int32)
  for i, n in enumerate(lens):
    m = -(-n // 64)
    bt[i, :m] = perm[at:at + m]
    at += m
    if n % 64:  # slots no token has written
      kc[bt[i, m - 1], :, n % 64:] = float("nan")
      vc[bt[i, m - 1], :, :, n % 64:] = float("inf")
  q = torch.randn(T, H, d, generator=g, device="cuda").bfloat16()
  pb = torch.randn(H, generator=g, device="cuda") - 2
  buf = torch.full((T, H * d + 8), 3.0, device="cuda", dtype=torch.bfloat16)
  out = buf[:, 4:4 + H * d]
  bt, cl, cu = bt.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda"), torch.arange(T + 1, dtype=torch.int32, device="cuda")
  K.attn_gated_chunk(q, kc, vc, bt, cu, cl, pb, d ** -0.5, chunk, 1.5, out, max_qlen=1)
  want = _exact(q, kc, vc, bt, lens, pb, d ** -0.5, chunk, 1.5)
  live = torch.tensor([n > 0 for n in lens], device="cuda")
  # fp32 throughout, then one rounding to bf16 (2^-9 of the result); scores and sums of at most 600 keys in fp32: well below it
  assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5)[live].all())
  assert float((buf[:, :4] - 3).abs().max()) == 0 and float((buf[:, -4:] - 3).abs().max()) == 0
  assert float((out[~live] - 3).abs().max()) == 0  # padding rows are not written


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,d", [(16, 4, 128), (16, 1, 64), (32, 4, 32), (12, 1, 96)])
@pytest.mark.parametrize("chunk,n", [(96, 130), (7, 60), (96, 100), (1024, 400)])
def test_values_that_are_no_numbers(H, G, d, chunk, n):
  """Values before the chunk that are no numbers or infinite, and those of keys whose weight underflowed, are left out; infinite ones
  of the chunk reach the sums of their channel with their sign, beside the terms of a weight that are 0."""
  g = torch.Generator(device="cuda").manual_seed(H + d + n)
  width, lo = -(-n // 64), (n - 1) // chunk * chunk
  kc = torch.randn(width, G, 64, d, generator=g, device="cuda").bfloat16()
  vc = torch.randn(width, G, d, 64, generator=g, device="cuda").bfloat16()
  q = torch.randn(1, H, d, generator=g, device="cuda").bfloat16()
  bt = torch.arange(width, dtype=torch.int32, device="cuda")[None].contiguous()
  cu, cl = torch.tensor([0, 1], dtype=torch.int32, device="cuda"), torch.tensor([n], dtype=torch.int32, device="cuda")

  def run(kc, vc, pb, max_qlen):
    out = torch.zeros(1, H * d, dtype=torch.bfloat16, device="cuda")
    K.attn_gated_chunk(q, kc, vc, bt, cu, cl, pb, d ** -0.5, chunk, 1.5, out, max_qlen=max_qlen)
    return out
  pb = torch.randn(H, generator=g, device="cuda") - 2
  plain = _exact(q, kc, vc, bt, [n], pb, d ** -0.5, chunk, 1.5)
  near = lambda got, want: bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all())  # noqa: E731 - (as above)
  if lo % 64:
    for bad in (float("nan"), float("-inf")):
      v = vc.clone()
      v[lo // 64, :, :, :lo % 64] = bad
      assert near(run(kc, v, pb, 1), plain), bad
  v = vc.clone()
  at = n - 1 - (n - 1 - lo) // 3  # a key of the chunk
  v[at // 64, :, 1, at % 64], v[at // 64, :, 5, at % 64], v[at // 64, :, 9, at % 64] = float("inf"), float("-inf"), float("nan")
  want = plain.view(1, H, d).clone()
  want[:, :, 1], want[:, :, 5], want[:, :, 9] = float("inf"), float("-inf"), float("nan")
  for max_qlen in (1, 0):  # (0: the kernel of any head size)
    got = run(kc, v, pb, max_qlen).double()
    same = ((got - want.view(1, -1)).abs() <= 2.0 ** -8 * want.view(1, -1).abs() + 1e-5) | (got == want.view(1, -1)) | (got.isnan() & want.view(1, -1).isnan())
    assert bool(same.all()), max_qlen
  off = torch.full_like(pb, -200.0)  # (every weight 0)
  for max_qlen in (1, 0):
    assert float(run(kc, v, off, max_qlen).abs().max()) == 0, max_qlen
