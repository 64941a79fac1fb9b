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
