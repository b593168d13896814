"""GPU parity of the expanded prompt path: mla_head_product_rows (cached
latents into each head's keys and values) and mla_prompt_attn (causal
attention over them), against fp64 on the CPU or GPU, and the rule that
routes a prompt there.

Bars: the products are rounded once, so every output lies within one bf16 ulp
of the exact one plus the fp32 summation bound K 2^-24 sum |x w|.  Attention
is compared with fp64 on the same bf16 keys, values and queries; its errors
are the bf16 weights (2^-9 relative each, so at most 2^-9 of sum_p |v| / sum_p
<= max |v|), the rotated queries (three bf16 roundings, a score error of at
most 3 * 2^-9 * scale * sum |q_pe k_pe|, which scales a weight by as much) and
the output's own rounding.
"""
import pytest
import torch

from swamla_amd import MLA, MLAConfig, kernels
from swamla_amd.kernels import LatentCache
from swamla_amd.rope import rope_tables

pytestmark = pytest.mark.gpu
SCALE = 192 ** -0.5


def say(*a):
    print(*a, flush=True)


def make_cache(B, S, rank, fp8, g, dev):
    cache = LatentCache.allocate(B, S, torch.bfloat16, dev, fp8=fp8, rank=rank)
    lat = torch.randn(B, S, rank, generator=g, device=dev).to(torch.bfloat16)
    if fp8:
        scale = lat.float().abs().amax(-1) / 448
        codes = (lat.float() / scale[..., None]).to(torch.float8_e4m3fn)
        cache.ckv[..., :rank] = codes.view(torch.uint8)
        cache.scale.copy_(scale)
        values = codes.double() * scale.double()[..., None]
    else:
        cache.ckv[..., :rank] = lat
        values = lat.double()
    cache.kpe.copy_(0.64 * torch.randn(B, S, 64, generator=g, device=dev))
    return cache, values


@pytest.mark.parametrize("fp8", [False, True], ids=["bf16", "fp8"])
@pytest.mark.parametrize("B,L,S,H,rank", [
    (1, 1, 1, 1, 64),        # one row, the narrowest rank, a group with idle waves
    (2, 33, 40, 3, 173),     # odd R_pad / 64, a partial tile in each sequence
    (3, 700, 701, 5, 256),   # several tiles per workgroup, partial last ones
    (1, 1031, 1031, 16, 320),
    (2, 257, 300, 4, 512),
    (1, 130, 130, 2, 577),   # above 512: one workgroup per CU
    (2, 1100, 1100, 16, 1024),
])
def test_head_product_rows(gpu, B, L, S, H, rank, fp8):
    say(f"rows B={B} L={L} S={S} H={H} rank={rank} fp8={fp8}")
    g = torch.Generator(device=gpu).manual_seed(rank + L)
    cache, values = make_cache(B, S, rank, fp8, g, gpu)
    w = (0.05 * torch.randn(H, 128, rank, generator=g, device=gpu)).to(torch.bfloat16)
    out = torch.full((B, H, L + 2, 128), 7.0, dtype=torch.bfloat16, device=gpu)
    kernels.head_product(cache.ckv[:, None, :L], kernels.pad_rank(w, rank), out=out[:, :, :L],
                         scale=cache.scale[:, :L] if fp8 else None)
    torch.cuda.synchronize()
    x, wd = values[:, :L].cpu(), w.double().cpu()
    ref = torch.einsum("bsk,hnk->bhsn", x, wd)
    slack = torch.einsum("bsk,hnk->bhsn", x.abs(), wd.abs()) * (rank * 2.0 ** -24)
    err = (out[:, :, :L].double().cpu() - ref).abs()
    bad = err > 2.0 ** -7 * ref.abs() + slack
    assert not bool(bad.any()), f"{int(bad.sum())} / {bad.numel()}, max err {float(err.max()):.3e}"
    assert bool((out[:, :, L:] == 7.0).all())


@pytest.mark.parametrize("rope_abs", [False, True], ids=["chunk", "abs"])
@pytest.mark.parametrize("B,T,start,H", [
    (1, 1, 0, 1), (1, 2, 63, 2), (2, 31, 1, 3), (1, 64, 0, 16), (1, 65, 64, 2), (2, 127, 0, 2), (1, 128, 129, 1),
    (3, 129, 0, 5), (1, 300, 1000, 4), (2, 700, 3, 2),
])
def test_prompt_attention(gpu, B, T, start, H, rope_abs):
    """Edges of the 32-query waves, 64-token tiles and 128-query workgroups."""
    say(f"prompt B={B} T={T} start={start} H={H} rope_abs={rope_abs}")
    g = torch.Generator(device=gpu).manual_seed(7 * T + start)
    L, S = start + T, start + T + 5
    cache, _ = make_cache(B, S, 64, False, g, gpu)
    q = (0.8 * torch.randn(B * T, H, 200, generator=g, device=gpu)).to(torch.bfloat16)[:, :, :192]
    k, v = (torch.randn(B, H, L, 128, generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    cos, sin = (t.to(torch.bfloat16)[0, 0, :, :32].contiguous().to(gpu) for t in rope_tables(64, S))
    out = torch.full((B * T, H, 136), 7.0, dtype=torch.bfloat16, device=gpu)
    kernels.prompt_attention(q, cos, sin, k, v, cache, SCALE, start=start, tokens_per_seq=T, rope_abs=rope_abs,
                             out=out[:, :, :128])
    torch.cuda.synchronize()
    qd = q.double().view(B, T, H, 192).transpose(1, 2)
    r0 = start if rope_abs else 0
    c, s = cos[r0:r0 + T].double(), sin[r0:r0 + T].double()
    x1, x2 = qd[..., 128::2], qd[..., 129::2]
    qp = torch.stack([x1 * c - x2 * s, x2 * c + x1 * s], -1).flatten(-2)
    pe = cache.kpe[:, None, :L].double()
    sc = (qd[..., :128] @ k.double().transpose(-1, -2) + qp @ pe.transpose(-1, -2)) * SCALE
    mask = torch.arange(L, device=gpu)[None] > start + torch.arange(T, device=gpu)[:, None]
    p = torch.softmax(sc.masked_fill(mask, float("-inf")), -1)
    vd = v.double()[..., torch.argsort(kernels.prompt_value_order(gpu))]
    ref = p @ vd
    # |score error| <= e: weights off by a factor within e^(+-e), and their sum too
    e = (3 * 2.0 ** -9 * SCALE * (qp.abs() @ pe.abs().transpose(-1, -2))).amax(-1, keepdim=True)
    bound = (p @ vd.abs()) * (torch.expm1(2 * e) + 2 * 2.0 ** -9) + 2.0 ** -8 * ref.abs() + 1e-6
    got = out[:, :, :128].double().view(B, T, H, 128).transpose(1, 2)
    bad = (got - ref).abs() > bound
    assert not bool(bad.any()), f"{int(bad.sum())} / {bad.numel()}"
    assert bool((out[:, :, 128:] == 7.0).all())


@pytest.mark.parametrize("rank,H,cache,q_lora", [(256, 16, None, 0), (444, 12, None, 0), (173, 32, "fp8_e4m3", 0),
                                                 (1000, 16, "fp8_e4m3", 0), (640, 16, None, 160)])
@pytest.mark.parametrize("B,T,start,per_pass", [(3, 190, 0, 1), (2, 260, 70, 2)])
def test_module_routes_agree(gpu, rank, H, cache, q_lora, B, T, start, per_pass, monkeypatch):
    """A prompt through MLA.forward on either route, sequence groups of one
    and of all: outputs within the bf16 bar, the caches' bits equal."""
    say(f"routes rank={rank} H={H} cache={cache} B={B} T={T} start={start}")
    cfg = MLAConfig(n_embd=512, n_head=H, kv_lora_rank=rank, q_lora_rank=q_lora, max_batch_size=B, max_seq_len=400)
    m = MLA(cfg, cache_dtype=cache)
    g = torch.Generator().manual_seed(rank)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("weight") and "norm" not in name:
                p.copy_(torch.randn(p.shape, generator=g) * 0.03)
    m.eval().to(torch.bfloat16).to(gpu)
    m.EXPAND_BYTES = per_pass * 2 * H * (start + T) * 256
    x0 = torch.randn(B, max(start, 1), 512, generator=g).to(torch.bfloat16).to(gpu)
    x = torch.randn(B, T, 512, generator=g).to(torch.bfloat16).to(gpu)
    outs, caches = {}, {}
    for use in (True, False):
        monkeypatch.setattr(kernels, "use_expanded", lambda *a, **k: use)
        calls = []
        real = kernels.prompt_attention
        monkeypatch.setattr(kernels, "prompt_attention", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
        m.clear_cache()
        m.set_inference_mode(True)
        with torch.no_grad():
            if start:
                m.prefill_cache(x0, 0)
            outs[use] = m(x, start).double()
        torch.cuda.synchronize()
        monkeypatch.setattr(kernels, "prompt_attention", real)
        assert len(calls) == (-(-B // per_pass) if use else 0)
        caches[use] = (m.kv_cache.clone(), m.pe_cache.clone())
    assert all(torch.equal(a, b) for a, b in zip(caches[True], caches[False]))
    err = (outs[True] - outs[False]).abs()
    assert not bool((err > 1e-2 + 2e-2 * outs[False].abs()).any()), float(err.max())


def test_prompt_in_a_graph(gpu):
    """A captured prompt replays to the eager result."""
    m = MLA(MLAConfig(n_embd=512, max_batch_size=2, max_seq_len=700)).eval().to(torch.bfloat16).to(gpu)
    m.set_inference_mode(True)
    g = torch.Generator(device=gpu).manual_seed(3)
    x = torch.randn(2, 640, 512, generator=g, device=gpu).to(torch.bfloat16)
    assert kernels.use_expanded(2, 640, 0, 16, 256)
    with torch.no_grad():
        want = m(x, 0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = m(x, 0)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)


@pytest.mark.parametrize("rope_abs", [False, True], ids=["chunk", "abs"])
@pytest.mark.parametrize("B,T,start,H", [
    (1, 1, 0, 1), (2, 2, 31, 3), (1, 31, 0, 2), (1, 32, 0, 2), (3, 33, 33, 1), (1, 64, 191, 2), (1, 257, 0, 16),
    (2, 300, 700, 2),
])
def test_prompt_attention_f32(gpu, B, T, start, H, rope_abs):
    """Edges of the 32-query blocks, the 32-token tiles and the eight waves
    they are dealt to (fewer tiles than waves, one more than a round).  Every
    product and sum is fp32: a score's error is at most about 200 roundings of
    its terms (2^-24 each), a weight's twice that."""
    say(f"prompt f32 B={B} T={T} start={start} H={H} rope_abs={rope_abs}")
    g = torch.Generator(device=gpu).manual_seed(11 * T + start)
    L, S = start + T, start + T + 3
    cache = LatentCache.allocate(B, S, torch.float32, gpu, rank=64)
    cache.kpe.copy_(torch.randn(B, S, 64, generator=g, device=gpu))
    q = (0.8 * torch.randn(B * T, H, 196, generator=g, device=gpu))[:, :, :192]
    kv = torch.randn(B, L, H, 256, generator=g, device=gpu)
    cos, sin = (t[0, 0, :, :32].contiguous().to(gpu) for t in rope_tables(64, S))
    out = torch.full((B * T, H, 132), 7.0, device=gpu)
    kernels.prompt_attention_f32(q, cos, sin, kv, cache, SCALE, start=start, tokens_per_seq=T, rope_abs=rope_abs,
                                 out=out[:, :, :128])
    torch.cuda.synchronize()
    qd = q.double().view(B, T, H, 192).transpose(1, 2)
    r0 = start if rope_abs else 0
    c, s = cos[r0:r0 + T].double(), sin[r0:r0 + T].double()
    x1, x2 = qd[..., 128::2], qd[..., 129::2]
    qd = torch.cat([qd[..., :128], torch.stack([x1 * c - x2 * s, x2 * c + x1 * s], -1).flatten(-2)], -1)
    kd = torch.cat([kv[..., :128].transpose(1, 2), cache.kpe[:, None, :L].expand(B, H, L, 64)], -1).double()
    mask = torch.arange(L, device=gpu)[None] > start + torch.arange(T, device=gpu)[:, None]
    p = torch.softmax((qd @ kd.transpose(-1, -2) * SCALE).masked_fill(mask, float("-inf")), -1)
    vd = kv[..., 128:].transpose(1, 2).double()
    ref = p @ vd
    e = 200 * 2.0 ** -24 * SCALE * (qd.abs() @ kd.abs().transpose(-1, -2)).amax(-1, keepdim=True)
    bound = (p @ vd.abs()) * (2 * e + L * 2.0 ** -24)
    got = out[:, :, :128].double().view(B, T, H, 128).transpose(1, 2)
    assert bool(((got - ref).abs() <= bound).all()), float(((got - ref).abs() / bound).max())
    assert bool((out[:, :, 128:] == 7.0).all())


@pytest.mark.parametrize("rank,H", [(256, 16), (173, 12)])
def test_module_f32_routes_agree(gpu, rank, H, monkeypatch):
    """An fp32 prompt and a chunk behind it on either route: equal to fp32
    sums in another order (1e-5 of the output's scale), cache bits equal."""
    cfg = MLAConfig(n_embd=512, n_head=H, kv_lora_rank=rank, max_batch_size=2, max_seq_len=260)
    m = MLA(cfg)
    g = torch.Generator().manual_seed(rank)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("weight") and "norm" not in name:
                p.copy_(torch.randn(p.shape, generator=g) * 0.03)
    m.eval().to(gpu)
    x0, x1 = (torch.randn(2, t, 512, generator=g).to(gpu) for t in (200, 45))
    outs = {}
    for use in (True, False):
        monkeypatch.setattr(kernels, "use_expanded_f32", lambda *a, **k: use)
        m.clear_cache()
        m.set_inference_mode(True)
        with torch.no_grad():
            outs[use] = [m(x0, 0), m(x1, 200), m.kv_cache.clone()]
    torch.cuda.synchronize()
    for a, b in zip(outs[True], outs[False]):
        assert float((a.double() - b.double()).abs().max()) <= 1e-5 * float(b.abs().max())
    assert torch.equal(outs[True][2], outs[False][2])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("where", ["v", "k", "pe"])
@pytest.mark.parametrize("T,start,bad", [(200, 0, 1), (200, 0, 199), (65, 30, 40), (300, 100, 128), (40, 2, 31)])
def test_later_nonfinite_tokens_stay_out(gpu, dtype, where, T, start, bad):
    """A token's infinities and NaN reach the rows that attend to it and no
    earlier one, at the edges of tiles and waves.  The clean rows are held to
    the bounds of test_prompt_attention / test_prompt_attention_f32, in the
    channels that hold no such value every row is."""
    say(f"non-finite {where} {dtype} T={T} start={start} bad={bad}")
    B, H = 2, 3
    bf = dtype == torch.bfloat16
    g = torch.Generator(device=gpu).manual_seed(T + bad)
    L, S, tok = start + T, start + T + 3, start + bad
    cache = LatentCache.allocate(B, S, dtype, gpu, rank=64)
    cache.kpe.copy_(0.64 * torch.randn(B, S, 64, generator=g, device=gpu))
    q = (0.8 * torch.randn(B * T, H, 192, generator=g, device=gpu)).to(dtype)
    k, v = (torch.randn(B, H, L, 128, generator=g, device=gpu).to(dtype) for _ in range(2))
    cos, sin = (t.to(dtype)[0, 0, :, :32].contiguous().to(gpu) for t in rope_tables(64, S))

    qd = q.double().view(B, T, H, 192).transpose(1, 2)
    c, s = cos[:T].double(), sin[:T].double()
    x1, x2 = qd[..., 128::2], qd[..., 129::2]
    qd = torch.cat([qd[..., :128], torch.stack([x1 * c - x2 * s, x2 * c + x1 * s], -1).flatten(-2)], -1)
    kd = torch.cat([k, cache.kpe[:, None, :L].expand(B, H, L, 64)], -1).double()
    mask = torch.arange(L, device=gpu)[None] > start + torch.arange(T, device=gpu)[:, None]
    p = torch.softmax((qd @ kd.transpose(-1, -2) * SCALE).masked_fill(mask, float("-inf")), -1)
    ref, spread = p @ v.double(), p @ v.double().abs()
    if bf:
        e = (3 * 2.0 ** -9 * SCALE * (qd[..., 128:].abs() @ kd[..., 128:].abs().transpose(-1, -2))).amax(-1, True)
        bound = spread * (torch.expm1(2 * e) + 2 * 2.0 ** -9) + 2.0 ** -8 * ref.abs() + 1e-6
    else:
        e = 200 * 2.0 ** -24 * SCALE * (qd.abs() @ kd.abs().transpose(-1, -2)).amax(-1, True)
        bound = spread * (2 * e + L * 2.0 ** -24)

    hit = torch.zeros(B, H, T, 128, dtype=torch.bool, device=gpu)  # what the planted values may reach
    if where == "v":
        v[:, :, tok, 5::16] = float("inf")
        v[:, :, L - 1, 6::16] = float("nan")
        hit[:, :, bad:, 5::16] = True
        hit[:, :, -1, 6::16] = True
    else:
        (k[:, :, tok] if where == "k" else cache.kpe[:, tok])[..., 3] = float("nan")
        hit[:, :, bad:] = True
    if bf:
        out = kernels.prompt_attention(q, cos, sin, k, v[..., kernels.prompt_value_order(gpu)].contiguous(), cache,
                                       SCALE, start=start, tokens_per_seq=T)
    else:
        out = kernels.prompt_attention_f32(q, cos, sin, torch.cat([k, v], -1).transpose(1, 2).contiguous(), cache,
                                           SCALE, start=start, tokens_per_seq=T)
    torch.cuda.synchronize()
    got = out.double().view(B, T, H, 128).transpose(1, 2)
    assert not bool(torch.isfinite(got[hit]).any())
    assert bool(((got - ref).abs() <= bound)[~hit].all()), float(((got - ref).abs() - bound)[~hit].max())


@pytest.mark.parametrize("dtype,cache,H", [(torch.bfloat16, None, 12), (torch.bfloat16, "fp8_e4m3", 16),
                                           (torch.float32, None, 12)])
@pytest.mark.parametrize("heads_at_once", [11, 8, 5, 1])
def test_expansion_in_head_groups(gpu, dtype, cache, H, heads_at_once, monkeypatch):
    """With less room than one sequence's keys and values need, heads go in
    groups that fit it: bf16 output bits as in one piece (fp32: another GEMM
    shape, 1e-5 of the scale)."""
    say(f"head groups {dtype} cache={cache} H={H} at once={heads_at_once}")
    B, T, start = 2, 300, 200
    m = MLA(MLAConfig(n_embd=512, n_head=H, max_batch_size=B, max_seq_len=512), cache_dtype=cache)
    g = torch.Generator().manual_seed(H)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("weight") and "norm" not in name:
                p.copy_(torch.randn(p.shape, generator=g) * 0.03)
    m.eval().to(dtype).to(gpu)
    m.set_inference_mode(True)
    per_head = 2 * (start + T) * 128 * (2 if dtype == torch.bfloat16 else 4)
    name = "prompt_attention" if dtype == torch.bfloat16 else "prompt_attention_f32"
    calls, real = [], getattr(kernels, name)

    def spy(q, cos, sin, *kv_cache, **k):
        room = sum(t.numel() * t.element_size() for t in kv_cache if isinstance(t, torch.Tensor))
        assert room <= m.EXPAND_BYTES
        calls.append(q.shape[1])
        return real(q, cos, sin, *kv_cache, **k)

    monkeypatch.setattr(kernels, name, spy)
    monkeypatch.setattr(kernels, "use_expanded", lambda *a, **k: True)
    monkeypatch.setattr(kernels, "use_expanded_f32", lambda *a, **k: True)
    x0, x = (torch.randn(B, t, 512, generator=g).to(dtype).to(gpu) for t in (start, T))
    outs = []
    for room in (B * H * per_head, heads_at_once * per_head + per_head // 2):
        m.EXPAND_BYTES = room
        calls.clear()
        with torch.no_grad():
            m.prefill_cache(x0, 0)
            outs.append(m(x, start))
        torch.cuda.synchronize()
        if len(outs) == 1:
            assert calls == [H]
    step = 8 if 8 < heads_at_once < 16 else heads_at_once
    assert calls == B * [min(step, H - h) for h in range(0, H, step)], calls
    if dtype == torch.bfloat16:
        assert torch.equal(*outs)
    else:
        assert float((outs[0] - outs[1]).abs().max()) <= 1e-5 * float(outs[0].abs().max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_no_room_for_the_expansion(gpu, dtype, monkeypatch):
    """No room for one head's keys and values, by EXPAND_BYTES or on the
    device: the call is the latent route's, bit for bit."""
    m = MLA(MLAConfig(n_embd=512, max_batch_size=1, max_seq_len=400))
    g = torch.Generator().manual_seed(9)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("weight") and "norm" not in name:
                p.copy_(torch.randn(p.shape, generator=g) * 0.03)
    m.eval().to(dtype).to(gpu)
    m.set_inference_mode(True)
    x = torch.randn(1, 400, 512, generator=g).to(dtype).to(gpu)
    rule = "use_expanded" if dtype == torch.bfloat16 else "use_expanded_f32"
    with torch.no_grad():
        monkeypatch.setattr(kernels, rule, lambda *a, **k: False)
        want = m(x, 0)
        monkeypatch.setattr(kernels, rule, lambda *a, **k: True)
        expanded = m(x, 0)
        m.EXPAND_BYTES = 1000
        assert torch.equal(m(x, 0), want)
        m.EXPAND_BYTES = MLA.EXPAND_BYTES
        assert torch.equal(m(x, 0), expanded)

        def full(*a, **k):
            raise torch.OutOfMemoryError("planted")

        monkeypatch.setattr(kernels, "head_product" if dtype == torch.bfloat16 else "prompt_attention_f32",
                            lambda x, *a, real=kernels.head_product, **k: real(x, *a, **k) if x.dim() == 3 and
                            dtype == torch.bfloat16 else full())
        assert torch.equal(m(x, 0), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_query_rows_of_any_alignment(gpu, dtype):
    """A query projection put in wq's place may return a view at any address."""

    class Offset(torch.nn.Linear):
        def forward(self, x):
            y = super().forward(x)
            out = torch.zeros(*y.shape[:-1], y.shape[-1] + 3, dtype=y.dtype, device=y.device)
            out[..., 3:] = y
            return out[..., 3:]

    m = MLA(MLAConfig(n_embd=512, kv_lora_rank=640, max_batch_size=1, max_seq_len=512)).eval().to(dtype).to(gpu)
    m.set_inference_mode(True)
    x = torch.randn(1, 512, 512, device=gpu).to(dtype)
    with torch.no_grad():
        want = m(x, 0)
        m.wq.__class__ = Offset
        assert torch.equal(m(x, 0), want)
