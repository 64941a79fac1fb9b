"""A decode step's inputs in one buffer, and the embedding rows of mixed-layer models in one launch."""
import pytest
import torch

from xotorch_support_jetson_amd.ops import kernels as K
from xotorch_support_jetson_amd.runtime.runner import _pack_layout, _unpack


@pytest.mark.parametrize("Bp,w", [(1, 1), (1, 8), (3, 5), (24, 32), (512, 129)])
def test_packed_inputs_do_not_overlap(Bp, w):
  layout, n = _pack_layout(Bp, w)
  buf = torch.zeros(n, dtype=torch.uint8)
  v = _unpack(buf, Bp, w)
  for i, (name, t) in enumerate(v.items()):
    assert layout[name][0] % 16 == 0 and t.shape == layout[name][2]
    t.fill_(i + 1)
  for i, t in enumerate(v.values()):
    assert bool((t == i + 1).all())
  big = torch.zeros(_pack_layout(Bp + 1, w + 1)[1], dtype=torch.uint8)  # a smaller step lies inside a larger one's buffer
  assert n <= big.numel() and set(_unpack(big, Bp, w)) == set(v)


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("D,V", [(1, 1), (4, 7), (30, 9), (1028, 50)])
@pytest.mark.parametrize("dt", [torch.int32, torch.int64])
def test_embedding_rows(dev, D, V, dt):
  table = torch.randn(V, D, generator=torch.Generator().manual_seed(D)).to(dev)
  ids = torch.tensor([0, V - 1, V, -1, 3 % V, 2 ** 31 - 1, -2 ** 31], dtype=dt).to(dev)
  want = table[ids.long().clamp(0, V - 1)]
  h, none = K.embed_rows(ids, table)
  h2, got = K.embed_rows(ids, table, want_ids=True)
  assert torch.equal(h, want) and torch.equal(h2, want) and none is None
  assert got.dtype == torch.int32 and torch.equal(got.long(), ids.long().clamp(0, V - 1))


def test_decode_steps_read_the_packed_inputs():
  """Decode steps through a stand-in for the captured graph: the same logits as steps without one, over growing and shrinking
  batches of a padded bucket and two table widths."""
  from xotorch_support_jetson_amd.inference.shard import Shard
  from xotorch_support_jetson_amd.models.config import PRESETS
  from xotorch_support_jetson_amd.runtime import runner as R
  for model in ("tiny-llama-d64", "tiny-tarepel"):
    c = PRESETS[model]
    plain, packed = (R.ShardRunner(c, Shard(model, 0, c.num_layers - 1, c.num_layers), "cpu", max_batch=6, max_ctx=640, num_pages=64,
                                   use_graphs=False) for _ in range(2))

    class Graph:
      def __init__(self, replay):
        self.replay = replay

    def capture(Bp, w):
      pack = torch.zeros(_pack_layout(Bp, w)[1], dtype=torch.uint8)
      g = {"pack": pack, **_unpack(pack, Bp, w), "x": torch.zeros(Bp, dtype=torch.int32)}
      inp = R.StepInputs(g["pos"], g["slots"], g["tables"], g["ctx"], torch.arange(Bp + 1, dtype=torch.int32), torch.arange(Bp), 1, True,
                         all_rows=True, state_slots=g["sslots"] if packed.sm is not None else None)
      g["graph"] = Graph(lambda: g.__setitem__("out", packed.model.forward(g["x"], inp)))
      packed._graphs[(Bp, w)] = g
      return g
    packed._capture, packed.use_graphs = capture, True
    for rids, lens in [("abc", [5, 70, 9]), ("abc", [1, 1, 1]), ("ac", [1, 1]), ("b", [1]), ("b", [500]), ("abc", [1, 1, 1])]:
      x = torch.randint(0, c.vocab_size, (sum(lens),), generator=torch.Generator().manual_seed(sum(lens)))
      # (padding rows change the products' shapes, so the last bits of their sums)
      torch.testing.assert_close(packed.forward(list(rids), lens, x), plain.forward(list(rids), lens, x), rtol=1e-2, atol=1e-2)
    assert len({w for _, w in packed._graphs}) == 2
