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
        for register in (m.resid_dropout.register_forward_hook, m.resid_dropout.register_forward_pre_hook):
            seen.clear()
            handle = register(lambda mod, *a: seen.append(mod))
            m(x, 0)
            handle.remove()
            assert seen == [m.resid_dropout]
        m.resid_dropout.forward = lambda x: 0.25 * x
        assert torch.equal(m(x, 0), 0.25 * want)
        del m.resid_dropout.forward
        assert torch.equal(m(x, 0), want)
        m.resid_dropout = type("Sub", (nn.Dropout,), {"forward": lambda self, x: 2 * x})()
        assert torch.equal(m.eval()(x, 0), 2 * want)
        m.resid_dropout = Halve()
        got = m(x, 0)
    torch.cuda.synchronize()
    assert torch.equal(got, 0.5 * want)


@pytest.mark.parametrize("q_lora", [0, 160])
def test_wide_step_calls_hooked_and_replaced_layers(gpu, q_lora, monkeypatch):
    """Above rank 512 a decode step's projections may be wrapped: hooks on
    them run, and a layer of another class with a weight of its own keeps its
    own forward.  Plain layers take the step's own launches."""
    say(f"wide step, hooks and replacements, q_lora={q_lora}")
    m, x = layer(gpu, 2, kv_lora_rank=640, q_lora_rank=q_lora), hidden(gpu, 3, 1)
    launches = []
    real = kernels.merge_project_wide
    monkeypatch.setattr(kernels, "merge_project_wide", lambda *a, **k: (launches.append(1), real(*a, **k))[1])
    names = ["wkv_a", "wo"] + (["wq"] if q_lora == 0 else ["wq_a", "q_norm", "wq_b"])
    with torch.no_grad():
        m.prefill_cache(hidden(gpu, 3, 50), 0)
        want = m(x, 50)
        assert len(launches) == 1
        for name in names:
            seen = []
            lin = getattr(m, name)
            for register in (lin.register_forward_hook, lin.register_forward_pre_hook):
                handle = register(lambda mod, *a: seen.append(mod))
                got = m(x, 50)
                handle.remove()
                assert seen == [lin], name
                seen.clear()
            err = (got.double() - want.double()).abs()
            assert not bool((err > 1e-2 + 2e-2 * want.double().abs()).any()), name

        class Doubled(type(m.wo)):
            def forward(self, x):
                return 2 * super().forward(x)

        plain, m.wo = m.wo, Doubled(*reversed(m.wo.weight.shape), bias=False).to(BF).to(gpu)
        m.wo.load_state_dict(plain.state_dict())
        err = (m(x, 50).double() - 2 * want.double()).abs()
        assert not bool((err > 2e-2 + 2e-2 * 2 * want.double().abs()).any())
        m.wo = plain
        launches.clear()
        assert torch.equal(m(x, 50), want) and len(launches) == 1


def misplace(m, names):
    """Parameters moved into one flat buffer, 2-byte aligned only."""
    ps = [p for n, p in m.named_parameters() if n.startswith(names)]
    buf = torch.empty(sum(p.numel() + 9 for p in ps), dtype=ps[0].dtype, device=ps[0].device)
    at = 1
    for p in ps:
        view = buf[at:at + p.numel()].view(p.shape)
        view.copy_(p.data)
        p.data = view
        at += p.numel()
        at += 1 + -at % 8
    assert ps and all(p.data_ptr() % 16 == 2 for p in ps)


@pytest.mark.parametrize("rank,q_lora,heads", [(640, 0, 16), (640, 100, 16), (640, 128, 12), (1000, 160, 16)])
@pytest.mark.parametrize("T", [1, 300])
def test_parameters_and_inputs_in_any_layout(gpu, rank, q_lora, heads, T):
    """Above rank 512, where steps and prompts were ATen products that take
    any layout: parameters at odd addresses (a prompt's own GEMMs keep
    aligned ones: only wkv_b is moved), a q_lora_rank the kernels' widths do
    not divide, and inputs that are misaligned, expanded or transposed views
    give what aligned ones give."""
    say(f"layouts rank={rank} q_lora={q_lora} heads={heads} T={T}")
    m = layer(gpu, 3, kv_lora_rank=rank, q_lora_rank=q_lora, n_head=heads)
    x, start = hidden(gpu, 2, T), 40 if T == 1 else 0

    with torch.no_grad():
        m.prefill_cache(hidden(gpu, 2, 40), 0)
        want = m(x, start)
        if T == 1:
            wide = torch.zeros(2, T, 515, dtype=BF, device=gpu)
            wide[:, :, 3:] = x
            assert torch.equal(m(wide[:, :, 3:], start), want)
        assert torch.equal(m(x.transpose(0, 2).contiguous().transpose(0, 2), start), want)
        assert torch.equal(m(x[:1].expand(2, T, 512), start), m(x[:1].repeat(2, 1, 1), start))
        misplace(m, ("w", "q_norm", "kv_norm") if T == 1 else ("wkv_b",))
        assert torch.equal(m(x, start), want)
        if q_lora and T == 1:
            with torch.autocast("cuda", dtype=BF):
                got = m(x, start)
            assert float((got.double() - want.double()).abs().max()) <= 1e-2 + 2e-2 * float(want.abs().max())
