"""The two statements of prompt_attention's value order agree (CPU)."""
import torch

from swamla_amd import kernels


def test_value_order():
    w = torch.arange(2 * 128 * 3).view(2, 128, 3)
    order = kernels.prompt_value_order()
    assert sorted(order.tolist()) == list(range(128))
    assert torch.equal(kernels.to_prompt_value_order(w), w[:, order])
