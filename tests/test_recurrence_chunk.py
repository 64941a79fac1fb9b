"""linear_recurrence in chunks of 16 tokens (csrc/recurrence_chunk.hip) against the recurrence token by token in float64: every
rule it takes, ends of chunks and of the ring of chunks in flight, decays at their extremes, channels and slots left alone."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.ops._ext import require

F64 = torch.float64
# rule -> (decay per key channel, delta rule, input scale, normaliser channel)
RULES = {"delta": (False, True, False, False), "channel_delta": (True, True, False, False), "channel": (True, False, False, False),
         "head": (False, False, False, False), "scaled": (False, False, True, False), "normaliser": (False, False, True, True)}


def token_by_token(q, k, v, decay, beta, q_scale, S, rule, H):
  """One sequence in float64: q, k [n, G, d], v [n, H, dvin], decay [n, H, d | 1], S [H, dv, d] -> (out [n, H, dv], S)."""
  _, delta, scaled, norm = RULES[rule]
  rep, out = H // q.shape[1], []
  for t in range(q.shape[0]):
    qt, kt = ((x[t].to(F64)).repeat_interleave(rep, 0) for x in (q, k))
    vt = v[t].to(F64)
    if norm:
      vt = torch.cat([vt, torch.ones(H, 1, dtype=F64)], 1)
    S = S * decay[t].to(F64)[:, None, :]
    if delta:
      vt = vt - torch.einsum("hvd,hd->hv", S, kt)
    if delta or scaled:
      vt = vt * beta[t].to(F64)[:, None]
    S = S + vt[:, :, None] * kt[:, None, :]
    out.append(torch.einsum("hvd,hd->hv", S, qt) * q_scale)
  return torch.stack(out), S


@pytest.mark.gpu
@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("d,dv,G", [(64, 40, 4), (128, 64, 2), (128, 17, 4)])
@pytest.mark.parametrize("decays", ["near one", "wide", "zero and above one"])
def test_chunks_match_token_by_token(gpu, rule, d, dv, G, decays):
  channel, delta, scaled, norm = RULES[rule]
  H, q_scale = 4, 0.7
  G = H if channel and not delta else G
  lens = [1, 15, 16, 17, 33, 100, 47]
  T, B, dvs = sum(lens), len(lens), dv + norm
  g = torch.Generator().manual_seed(d + dv + len(rule))
  rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
  q, k, v = rn(T, G, d), rn(T, G, d), rn(T, H, dv)
  q, k = q / q.norm(dim=-1, keepdim=True), k / k.norm(dim=-1, keepdim=True)
  a = rn(T, H, d if channel else 1)
  if decays == "near one":
    a = torch.sigmoid(3 + a) ** (1 / 16)
  elif decays == "wide":
    a = torch.exp(-3 * torch.nn.functional.softplus(3 * a))
  else:
    a = torch.where(a > 1, torch.zeros_like(a), torch.where(a < -1.5, torch.full_like(a, 1.1), torch.sigmoid(a + 2)))
  beta = torch.sigmoid(rn(T, H)) if delta else torch.rand(T, H, generator=g) * 2 if scaled else None
  state = rn(B + 2, H, dvs, d)
  slots = torch.tensor([3, -1, 5, 0, 8, 1, 6], dtype=torch.int32)
  cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
  S, out = state.to(gpu), torch.full((T, H * dvs), 7.0, device=gpu)
  # (q and k as column slices of wider rows)
  wide = torch.zeros(T, 2 * G * d + 8)
  wide[:, 4:4 + G * d], wide[:, 4 + G * d:4 + 2 * G * d] = q.reshape(T, -1), k.reshape(T, -1)
  wide = wide.to(gpu)
  K.linear_recurrence(wide[:, 4:4 + G * d], wide[:, 4 + G * d:4 + 2 * G * d], v.reshape(T, -1).to(gpu), a.reshape(T, -1).to(gpu),
                      None if beta is None else beta.to(gpu), q_scale, S, slots.to(gpu), cu.to(gpu), out, plain=scaled and not norm, max_qlen=100)
  S, out = S.cpu(), out.cpu().view(T, H, dvs)
  kept = [s for s in range(B + 2) if s not in slots.tolist()]
  assert torch.equal(S[kept], state[kept])
  for b in range(B):
    t0, t1, slot = int(cu[b]), int(cu[b + 1]), int(slots[b])
    if slot < 0:
      assert (out[t0:t1] == 7.0).all()
      continue
    want, last = token_by_token(q[t0:t1], k[t0:t1], v[t0:t1], a[t0:t1], None if beta is None else beta[t0:t1], q_scale,
                                state[slot].to(F64), rule, H)
    # fp32 products and sums throughout: dot products of d and of 16 terms and a chain of at most 100 decays and writes, a
    # few units of 6e-8 each (the token-by-token kernel: 1e-7 to 3e-7)
    for got, ref in ((out[t0:t1], want), (S[slot], last)):
      assert ((got.to(F64) - ref).norm() / ref.norm()) < 1e-6, (b, lens[b])


@pytest.mark.gpu
@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lens", [(100, 97, 96, 1, 112, 95, 81, 60), (97, 33, 16) * 6], ids=["halves", "many"])
def test_forms_of_the_scan(gpu, rule, d, lens):
  """Steps bound by all their chunks (csrc/recurrence_chunk.hip go()): waves of half of the key dims, with two chunks and, the delta rule's
  of more than 512 workgroups, with one in flight; the other tests' steps are bound by their longest sequence."""
  channel, delta, scaled, norm = RULES[rule]
  H, dv, q_scale = 16, 64 - norm, 0.7
  G = H if channel and not delta else 4
  T, B, dvs = sum(lens), len(lens), dv + norm
  assert T * H * 2 >= 180 * max(lens) and (B * H * 2 > 512) == (B > 16)
  g = torch.Generator().manual_seed(d + B)
  rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
  q, k, v, a = rn(T, G, d), rn(T, G, d), rn(T, H, dv), torch.sigmoid(3 + rn(T, H, d if channel else 1)) ** (1 / 16)
  q, k = q / q.norm(dim=-1, keepdim=True), k / k.norm(dim=-1, keepdim=True)
  beta = torch.sigmoid(rn(T, H)) if delta or scaled else None
  state, cu = rn(B, H, dvs, d), torch.tensor((0, *lens)).cumsum(0).to(torch.int32)

  def run(v):
    S, out = state.to(gpu), torch.full((T, H * dvs), 7.0, device=gpu)
    K.linear_recurrence(*(x.reshape(T, -1).to(gpu) for x in (q, k, v, a)), None if beta is None else beta.to(gpu), q_scale, S,
                        torch.arange(B, dtype=torch.int32, device=gpu), cu.to(gpu), out, plain=scaled and not norm, max_qlen=max(lens))
    return S.cpu(), out.cpu().view(T, H, dvs)
  S, out = run(v)
  for b in range(min(B, 7)):
    t0, t1 = int(cu[b]), int(cu[b + 1])
    want, last = token_by_token(q[t0:t1], k[t0:t1], v[t0:t1], a[t0:t1], None if beta is None else beta[t0:t1], q_scale,
                                state[b].to(F64), rule, H)
    for got, ref in ((out[t0:t1], want), (S[b], last)):  # (the bound of test_chunks_match_token_by_token)
      assert ((got.to(F64) - ref).norm() / ref.norm()) < 1e-6, (b, lens[b])
  v[44, 3, 5] = float("nan")  # (a token of the first sequence: what is not behind it, and other heads, as without it)
  S2, out2 = run(v)
  other = [h for h in range(H) if h != 3]
  torch.testing.assert_close(out2[:44], out[:44], rtol=0, atol=float(2e-6 * out[:44].abs().max()))
  assert out2[44, 3, 5].isnan() and torch.equal(out2[:, other], out[:, other]) and torch.equal(out2[lens[0]:], out[lens[0]:])
  assert torch.equal(S2[1:], S[1:]) and torch.equal(S2[0, other], S[0, other])


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("rank", [16, 48, 24])
def test_decays_from_a_low_rank_product(gpu, d, rank):
  """linear_recurrence_made without A_log: decays of gla_prep, made by the chunks; a rank of no whole 16 is left to the two launches."""
  H, dv, tau, lens = 2, 33, 16.0, [101, 16, 1, 47]
  T, B, off = sum(lens), len(lens), 8
  g = torch.Generator().manual_seed(d + rank)
  rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
  P, a2, a2_b = rn(T, off + rank + 4), rn(H * d, rank) / rank ** 0.5, rn(H * d) + 3
  q, k, v, state = rn(T, H * d) / d ** 0.5, rn(T, H * d) / d ** 0.5, rn(T, H * dv), rn(B, H, dv, d)
  cu, slots = torch.tensor([0] + lens).cumsum(0).to(torch.int32), torch.arange(B, dtype=torch.int32)
  S, out = state.to(gpu), torch.full((T, H * dv), 7.0, device=gpu)
  took = require().linear_recurrence_made(q.to(gpu), k.to(gpu), v.to(gpu), P.to(gpu), off, a2.to(gpu), a2_b.to(gpu), tau, None, 0.7, S,
                                          slots.to(gpu), cu.to(gpu), out, max(lens))
  assert took == (rank % 16 == 0)
  if not took:
    assert (out == 7.0).all() and torch.equal(S.cpu(), state)
    return
  a = torch.exp(torch.nn.functional.logsigmoid(P[:, off:off + rank].to(F64) @ a2.to(F64).T + a2_b.to(F64)) / tau).view(T, H, d)
  S, out = S.cpu(), out.cpu().view(T, H, dv)
  for b in range(B):
    t0, t1 = int(cu[b]), int(cu[b + 1])
    want, last = token_by_token(*(x[t0:t1].view(t1 - t0, H, -1) for x in (q, k, v)), a[t0:t1], None, 0.7, state[b].to(F64), "channel", H)
    # fp32 sums of up to 48 products: some 3e-7 of |z| < 7, a sixteenth of it in a decay's logarithm, over the about 60 tokens that a decay
    # of 0.98 remembers: below 1e-5, the rest as in test_chunks_match_token_by_token
    for got, ref in ((out[t0:t1], want), (S[b], last)):
      assert ((got.to(F64) - ref).norm() / ref.norm()) < 1e-5, (b, lens[b])


@pytest.mark.gpu
@pytest.mark.parametrize("d,G", [(64, 2), (128, 4)])
def test_decays_and_write_strengths_from_finished_products(gpu, d, G):
  """linear_recurrence_made with A_log: exactly what recurrence_gates' decays and write strengths give, which are the same arithmetic."""
  H, dv, lens = 4, 40, [97, 33, 100, 1]
  T, B = sum(lens), len(lens)
  g = torch.Generator(device=gpu).manual_seed(d)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  P, za, dt_bias, A_log = rn(T, H + 3), rn(T, H * d + 8), rn(H * d), rn(H) * 0.4 - 1.2
  q, k, v, state = rn(T, G * d) / d ** 0.5, rn(T, G * d) / d ** 0.5, rn(T, H * dv), rn(B, H, dv, d)
  cu, slots = torch.tensor([0] + lens, device=gpu).cumsum(0).to(torch.int32), torch.arange(B, dtype=torch.int32, device=gpu)
  beta, decay = torch.empty(T, H, device=gpu), torch.empty(T, H * d, device=gpu)
  K.recurrence_gates(P, 2, beta, 0, None, dt_bias, A_log, decay, 0, None, None, za=za)
  one, two = (state.clone(), torch.empty(T, H * dv, device=gpu)), (state.clone(), torch.empty(T, H * dv, device=gpu))
  K.linear_recurrence(q, k, v, decay, beta, 0.7, one[0], slots, cu, one[1], max_qlen=100)
  assert require().linear_recurrence_made(q, k, v, P, 2, za, dt_bias, 1.0, A_log, 0.7, two[0], slots, cu, two[1], 100)
  assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])


ALL, SCALAR, NONE = {"delta", "channel_delta", "channel", "scaled"}, {"delta", "scaled"}, set()


@pytest.mark.gpu
@pytest.mark.parametrize("rule", sorted(ALL))
@pytest.mark.parametrize("B,dv,longest,chunks", [
  (1, 64, 55, NONE), (1, 64, 56, SCALAR), (3, 64, 63, SCALAR), (3, 64, 64, ALL), (4, 16, 64, ALL), (5, 32, 95, NONE), (5, 32, 96, ALL),  # prompts
  (32, 128, 31, NONE), (32, 128, 32, ALL), (31, 128, 32, NONE), (129, 128, 35, ALL), (129, 128, 31, NONE),  # that fill the CUs twice over, or nearly
  (16, 64, -55, NONE), (16, 64, -56, SCALAR), (17, 128, -95, NONE), (17, 128, -96, ALL), (32, 64, -64, ALL),  # (minus: behind single tokens)
  (64, 128, -47, NONE), (64, 128, -48, ALL), (56, 64, -95, NONE), (128, 128, -63, NONE), (128, 128, -64, ALL), (129, 128, -95, NONE),
  (136, 128, -95, NONE), (136, 128, -96, ALL)])
def test_both_sides_of_the_chunk_rule(gpu, rule, B, dv, longest, chunks):
  """The lengths from which steps go by chunks (mixers.hip chunks_take), against the same step token by token (longest taken as 1): the
  same numbers to the bit where the rule leaves it at that, sums in another order where it does not."""
  channel, delta, scaled, _ = RULES[rule]
  lens = [1] * (B - 1) + [-longest] if longest < 0 else [max(1, longest - 5 * b % longest) for b in range(B)]
  H, d, longest = 16, 64, max(lens)
  T, g = sum(lens), torch.Generator(device=gpu).manual_seed(B + longest)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  q, k, v, a = rn(T, H * d) / 8, rn(T, H * d) / 8, rn(T, H * dv), torch.sigmoid(3 + rn(T, H * (d if channel else 1)))
  beta, state = torch.sigmoid(rn(T, H)) if delta or scaled else None, rn(B, H, dv, d)
  slots, cu, got = torch.arange(B, dtype=torch.int32, device=gpu), torch.tensor([0] + lens).cumsum(0).int().to(gpu), []
  for said in (1, longest):
    S, out = state.clone(), torch.empty(T, H * dv, device=gpu)
    K.linear_recurrence(q, k, v, a, beta, 0.7, S, slots, cu, out, plain=scaled, max_qlen=said)
    got.append((out, S))
  for one, other in zip(*got):  # (both are within 1e-6 of float64, test_chunks_match_token_by_token; a single value within some times that)
    assert ((one - other).norm() / one.norm()) < 2e-6 and torch.equal(one, other) == (rule not in chunks)
    torch.testing.assert_close(one, other, rtol=0, atol=float(4e-6 * one.abs().max()))


@pytest.mark.gpu
def test_chunk_rule_keeps_what_it_cannot_take(gpu):
  """Rows off 16 bytes, key dims it has no tiles for and short steps run token by token, with the same results."""
  g = torch.Generator(device=gpu).manual_seed(3)
  T, H, dv = 130, 2, 24
  cu, slots = torch.tensor([0, T], dtype=torch.int32, device=gpu), torch.zeros(1, dtype=torch.int32, device=gpu)
  for d, off in ((64, 0), (64, 1), (48, 0)):
    x = torch.randn(T, 2 * H * d + off, device=gpu, generator=g) / d ** 0.5
    v, a, b = torch.randn(T, H * dv, device=gpu, generator=g), torch.rand(T, H, device=gpu, generator=g), torch.rand(T, H, device=gpu, generator=g)
    got = []
    for longest in (1, T):
      S, out = torch.zeros(1, H, dv, d, device=gpu), torch.empty(T, H * dv, device=gpu)
      K.linear_recurrence(x[:, off:off + H * d], x[:, off + H * d:], v, a, b, 1.0, S, slots, cu, out, max_qlen=longest)
      got.append((out, S))
    for one, other in zip(*got):
      torch.testing.assert_close(one, other, rtol=0, atol=float(2e-6 * one.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "decay", "beta"])
def test_a_value_that_is_no_number_reaches_no_earlier_token(gpu, rule, value, where):
  """Outputs before the token that holds it are those without it, and later ones are numbers wherever the recurrence token by
  token gives numbers (other channels, other heads, the other sequence)."""
  channel, delta, scaled, norm = RULES[rule]
  if where == "beta" and not (delta or scaled):
    pytest.skip("the rule has no input scale")
  g = torch.Generator().manual_seed(len(rule) + len(where))
  rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
  H, d, dv, lens = 2, 64, 40, [117, 100]
  T, dvs, t = sum(lens), dv + norm, 44  # token 12 of the first sequence's third chunk
  q, k, v, a = rn(T, H, d), rn(T, H, d), rn(T, H, dv), torch.rand(T, H, d if channel else 1, generator=g) * 0.2 + 0.8
  k = k / k.norm(dim=-1, keepdim=True)
  beta = torch.rand(T, H, generator=g) if delta or scaled else None
  bad = {"q": q, "k": k, "v": v, "decay": a, "beta": beta}
  one = {n: None if x is None else x.clone() for n, x in bad.items()}
  one[where][t, 1, ...] = value if where == "beta" else one[where][t, 1]
  if where != "beta":
    one[where][t, 1, 0] = value

  def run(x):
    S, out = torch.zeros(2, H, dvs, d, device=gpu), torch.empty(T, H * dvs, device=gpu)
    K.linear_recurrence(*(x[n].reshape(T, -1).to(gpu) for n in ("q", "k", "v", "decay")),
                        None if beta is None else x["beta"].to(gpu), 0.7, S, torch.tensor([0, 1], dtype=torch.int32, device=gpu),
                        torch.tensor([0, lens[0], T], dtype=torch.int32, device=gpu), out, plain=scaled and not norm, max_qlen=117)
    return out.cpu().view(T, H, dvs)
  clean, got = run(bad), run(one)
  torch.testing.assert_close(got[:t], clean[:t], rtol=0, atol=float(2e-6 * clean[:t].abs().max()))
  assert torch.equal(got[:, 0], clean[:, 0]) and torch.equal(got[lens[0]:], clean[lens[0]:])
  want, _ = token_by_token(*(one[n][:lens[0]] for n in ("q", "k", "v", "decay")), None if beta is None else one["beta"][:lens[0]],
                           0.7, torch.zeros(H, dvs, d, dtype=F64), rule, H)
  number = torch.isfinite(want)
  assert not number[t].all()
  diff = torch.where(number, got[:lens[0]].to(F64) - want, torch.zeros((), dtype=F64)).abs().max()
  assert diff < 1e-5 * want[number].abs().max()
  assert not torch.isfinite(got[:lens[0]][~number]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("rule,d,H,G,dv,lens", [("channel_delta", 128, 16, 16, 40, (9000, 3, 40, 7001, 4001)),  # 27 KB a chunk and head
                                               ("channel", 64, 32, 32, 33, (1, 9, 12100, 12001, 0, 3000)),
                                               ("delta", 64, 64, 2, 8, (31, 50000, 800, 17, 14003)), ("head", 64, 64, 1, 8, (70001,))])
def test_long_steps_go_in_portions_of_the_workspace(gpu, rule, d, H, G, dv, lens):
  """A step whose chunks' records are more than 512 MB, in portions of every sequence and (delta; the longest not known) of the slots: no
  more memory than that, and bit for bit the numbers of its sequences alone, token by token within the forms' bound."""
  channel, delta, _, _ = RULES[rule]
  T, B = sum(lens), len(lens)
  g = torch.Generator(device=gpu).manual_seed(T)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  q, k, v = rn(T, G * d) / d ** 0.5, rn(T, G * d) / d ** 0.5, rn(T, H * dv)
  a, beta = torch.sigmoid(3 + rn(T, H * (d if channel else 1))), torch.sigmoid(rn(T, H)) if delta else None
  state, starts = rn(B, H, dv, d), torch.tensor([0, *lens]).cumsum(0).tolist()

  def run(b0, b1, longest):
    t0, t1 = starts[b0], starts[b1]
    S, out = state[b0:b1].clone(), torch.full((t1 - t0, H * dv), 7.0, device=gpu)
    cu = torch.tensor([x - t0 for x in starts[b0:b1 + 1]], dtype=torch.int32, device=gpu)
    slots = torch.arange(b1 - b0, dtype=torch.int32, device=gpu)
    torch.cuda.synchronize()
    held = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    K.linear_recurrence(q[t0:t1], k[t0:t1], v[t0:t1], a[t0:t1], None if beta is None else beta[t0:t1], 0.7, S, slots, cu, out, max_qlen=longest)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - held <= (512 << 20) + (2 << 20)  # (blocks of 2 MB)
    return out, S
  out, S = run(0, B, max(lens))
  assert not out.isnan().any()
  for said in (0, T + 1, 1000):  # (fewer than there are: what is said chooses the way, not the numbers)
    assert all(torch.equal(x, y) for x, y in zip((out, S), run(0, B, said)))
  for b in range(B):
    if lens[b] >= 96:  # (shorter ones alone go token by token)
      one, last = run(b, b + 1, lens[b])
      assert torch.equal(out[starts[b]:starts[b + 1]], one) and torch.equal(S[b], last[0]), lens[b]
  for got, want in zip((out, S), run(0, B, 1)):  # (both within 1e-6 of float64, test_chunks_match_token_by_token)
    assert ((got - want).norm() / want.norm()) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("ld", [0, 4, 64])  # one row for all tokens, rows that overlap, rows whose heads lie in the next ones
def test_rows_that_repeat_or_overlap(gpu, rule, ld):
  """q, k and v of fewer floats a token than their heads hold: as the same rows one behind the other."""
  channel, delta, scaled, norm = RULES[rule]
  H, d, dv, lens = 4, 64, 40, [101, 17, 50]
  T, B = sum(lens), len(lens)
  g = torch.Generator(device=gpu).manual_seed(ld)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  q, k, v = ((rn(T * ld + H * n) / n ** 0.5).as_strided((T, H * n), (ld, 1)) for n in (d, d, dv))
  a, beta = torch.sigmoid(3 + rn(T, H * (d if channel else 1))), torch.sigmoid(rn(T, H)) if delta or scaled else None
  state, cu = rn(B, H, dv + norm, d), torch.tensor([0, *lens]).cumsum(0).int().to(gpu)
  slots, got = torch.arange(B, dtype=torch.int32, device=gpu), []
  for x in ((q, k, v), tuple(t.contiguous() for t in (q, k, v))):
    S, out = state.clone(), torch.full((T, H * (dv + norm)), 7.0, device=gpu)
    K.linear_recurrence(*x, a, beta, 0.7, S, slots, cu, out, plain=scaled and not norm, max_qlen=max(lens))
    got.append((out, S))
  assert all(torch.equal(one, other) for one, other in zip(*got))


@pytest.mark.gpu
@pytest.mark.parametrize("d,H,lens,made", [(64, 16, (200, 31, 1), True), (64, 15, (200, 31, 1), False), (128, 32, (450, 31), True), (128, 32, (400, 31), False),
                                          (64, 64, (31, 31, 31), False), (64, 16, (20,) * 32, False)])
def test_low_rank_decays_by_the_chunks_or_apart(gpu, d, H, lens, made, monkeypatch):
  """recurrence_norm with a low-rank decay: made by the chunks where these are many enough (16 chunk slots of 16 heads at key dims of 64,
  32 of 32 at 128) and a prompt is long enough for them, else in a launch of its own; the same numbers."""
  T, B, dv, rank, tau = sum(lens), len(lens), 32, 16, 16.0
  g = torch.Generator(device=gpu).manual_seed(T)
  rn = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
  P, a2, a2_b, qkv = rn(T, rank + 16), rn(H * d, rank) / rank ** 0.5, rn(H * d) + 3, rn(T, H * (2 * d + dv)) / d ** 0.5
  q, k, v = qkv[:, :H * d], qkv[:, H * d:2 * H * d], qkv[:, 2 * H * d:]
  state, w, gate, slots = rn(B, H, dv, d), rn(dv), rn(T, H * dv), torch.arange(B, dtype=torch.int32, device=gpu)
  cu, calls, C = torch.tensor([0, *lens], device=gpu).cumsum(0).int(), [], require()

  class Seen:
    def __getattr__(self, name):
      calls.append(name)
      return getattr(C, name)
  monkeypatch.setattr(K, "require", Seen)
  decay, got = torch.empty(T, H * d, device=gpu), []
  K.gla_prep(P, 8, a2, a2_b, tau, decay)
  for kw in (dict(gla=(P, 8, a2, a2_b, tau)), {}):
    calls.clear()
    S, out = state.clone(), torch.empty(T, H * dv, device=gpu)
    K.recurrence_norm(q, k, v, None if kw else decay, None, 0.7, S, slots, cu, w, gate, False, 1e-5, 1.0, out, max_qlen=max(lens), **kw)
    got.append((out, S))
    assert ("linear_recurrence_made" in calls) == (made and bool(kw)) and ("linear_recurrence" in calls) == (not made or not kw)
  # (the same to the bit apart; made by the chunks the low-rank sums are in another order: some 1e-7 of |z| < 7, a sixteenth of it in a decay's
  # logarithm, over the tokens that a decay remembers)
  for one, other in zip(*got):
    assert torch.equal(one, other) if not made else ((one - other).norm() / other.norm()) < 1e-5
