"""What MLA.forward owes the modules a user puts into it: their own forward
and their hooks, and parameters and inputs in any layout torch accepts."""
import pytest
import torch
import torch.nn as nn

from swamla_amd import MLA, MLAConfig, kernels

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def say(*a):
    print(*a, flush=True)


def layer(gpu, seed, dtype=BF, **kw):
    m = MLA(MLAConfig(n_embd=512, max_batch_size=3, max_seq_len=400, **kw))
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if "norm" not in name:
                p.copy_(torch.randn(p.shape, generator=g) * 0.03)
    m.eval().to(dtype).to(gpu)
    m.set_inference_mode(True)
    return m


def hidden(gpu, B, T, dtype=BF):
    g = torch.Generator().manual_seed(B + T)
    return torch.randn(B, T, 512, generator=g).to(dtype).to(gpu)


# (rank, tokens): the fused step, the step above rank 512, a prompt on each of
# the routes over expanded keys, and (fp32) a step
CALLS = [(256, 1, BF), (640, 1, BF), (256, 300, BF), (640, 300, BF), (256, 1, torch.float32), (256, 300, torch.float32)]


class Halve(nn.Module):
    def forward(self, x):
        return 0.5 * x


@pytest.mark.parametrize("rank,T,dtype", CALLS)
def test_resid_dropout_is_called(gpu, rank, T, dtype):
    """A module put in place of resid_dropout acts in eval, hooks on it and
    hooks on every module see its call."""
    say(f"resid_dropout rank={rank} T={T} {dtype}")
    m, x = layer(gpu, 1, dtype, kv_lora_rank=rank), hidden(gpu, 2, T, dtype)
    with torch.no_grad():
        want = m(x, 0)
        seen = []
        handle = nn.modules.module.register_module_forward_hook(lambda mod, a, out: seen.append(mod))
        try:
            m(x, 0)
        finally:
            handle.remove()
        assert m.resid_dropout in seen
        m.resid_dropout = Halve()
        got = m(x, 0)
    torch.cuda.synchronize()
    assert torch.equal(got, 0.5 * want)
