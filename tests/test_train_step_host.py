"""What a training step hands back to the host: its loss and the input gradient, which travels under the optimizer."""
import numpy as np
import pytest
import torch


@pytest.mark.gpu
def test_step_returns_this_steps_gradient(gpu):
  """The gradients of two steps stay what each step's backward gave (lr 0: the weights do not move); lengths as lists, arrays and
  tensors on either side, beyond the sequence too."""
  from xotorch_support_jetson_amd.inference.shard import Shard
  from xotorch_support_jetson_amd.models.config import PRESETS
  from xotorch_support_jetson_amd.runtime.runner import ShardRunner
  from xotorch_support_jetson_amd.train.trainer import ShardTrainer
  cfg = PRESETS["tiny-llama"]
  shard = Shard("tiny-llama", 1, cfg.num_layers - 1, cfg.num_layers)
  tr = ShardTrainer(ShardRunner(cfg, shard, gpu, max_batch=2, max_ctx=64).weights, gpu, lr=0.0)
  g = torch.Generator().manual_seed(0)
  y = torch.randint(0, cfg.vocab_size, (2, 24), generator=g)
  got = []
  for length in ([24, 9], np.array([24, 9]), torch.tensor([24, 9]), torch.tensor([24, 9], device=gpu), [80, 9]):
    x = torch.randn(2, 24, cfg.hidden_size, generator=g).to(torch.bfloat16)
    loss, grad = tr.step("r", x, y, length)
    tr.zero_grad()
    leaf, out = tr.forward_train(x)
    want_loss, want = tr.backward_accumulate(leaf, out, target=y, length=torch.as_tensor(np.asarray([24, 9])))
    assert grad.device.type == "cpu" and not grad.is_pinned() and loss == float(want_loss)
    got.append((grad, grad.clone(), want.cpu()))
  for grad, then, want in got:
    assert torch.equal(grad, then) and torch.equal(grad, want)
