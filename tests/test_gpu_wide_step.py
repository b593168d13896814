"""GPU parity of the decode step above rank 512: mla_merge_project_wide and
the module's step around it."""
import pytest
import torch

from attn_ref import wide_bars
from swamla_amd import MLA, MLAConfig, kernels
from swamla_amd.kernels import DecodeWorkspace, LatentCache
from swamla_amd.rope import rope_tables

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("n_splits,min_chunk,rank,rows", [
    (1, 64, 640, 5), (3, 64, 577, 33), (8, 64, 1024, 40), (47, 64, 1024, 9), (12, 64, 700, 40), (8, 64, 960, 70),
])
def test_merge_project_wide(gpu, n_splits, min_chunk, rank, rows):
    """Against mla_merge followed by the product in fp32, on ragged rows
    (empty, one and many splits in one call; two, four and eight rows per
    block, one and several merge groups).  Both merges round o_lat once to
    bf16 and may differ by an ulp of it (2^-7 |w| |o| summed), the output is
    rounded once (2^-8)."""
    say(f"wide merge n_splits={n_splits} rank={rank} rows={rows}")
    g = torch.Generator(device=gpu).manual_seed(rank + rows)
    rp, S = kernels.padded_rank(rank), 3000
    cache = LatentCache.allocate(rows, S, BF, gpu, rank=rank)
    cache.ckv[..., :rank] = torch.randn(rows, S, rank, generator=g, device=gpu)
    cache.kpe.copy_(torch.randn(rows, S, 64, generator=g, device=gpu))
    cos, sin = (t.to(BF)[0, 0, :, :32].contiguous().to(gpu) for t in rope_tables(64, S))
    sp = torch.randint(0, S, (rows,), generator=g, device=gpu, dtype=torch.int32)
    sp[:4] = torch.tensor([-1, 0, S - 1, 64], dtype=torch.int32)
    q_abs = (0.3 * torch.randn(rows, 16, rp, generator=g, device=gpu)).to(BF)
    q_pe = (0.3 * torch.randn(rows, 16, 64, generator=g, device=gpu)).to(BF)
    w_uv = kernels.pad_rank((0.05 * torch.randn(16, 128, rank, generator=g, device=gpu)).to(BF), rank)
    ws = DecodeWorkspace.allocate(rows, n_splits, gpu, rank=rank) if n_splits > 1 else None
    o_lat = torch.empty(rows, 16, rp, dtype=BF, device=gpu)
    kw = dict(start_pos=sp, n_splits=n_splits, min_chunk=min_chunk)
    kernels.decode_attention(q_abs, q_pe, cos, sin, cache, 0.0721, out=o_lat, workspace=ws, merge=False, **kw)
    got = torch.full((rows, 16, 128), float("nan"), dtype=BF, device=gpu)
    kernels.merge_project_wide(o_lat, w_uv, got, cache, workspace=ws, **kw)
    o_ref = kernels.decode_attention(q_abs, q_pe, cos, sin, cache, 0.0721, **kw)
    torch.cuda.synchronize()
    o, w = o_ref.double().cpu(), w_uv.double().cpu()
    ref = torch.einsum("rhc,hdc->rhd", o, w)
    bound = 2.0 ** -7 * torch.einsum("rhc,hdc->rhd", o.abs(), w.abs()) + 2.0 ** -8 * ref.abs()
    err = (got.double().cpu() - ref).abs()
    assert bool((err <= bound).all()), float((err - bound).max())
    assert bool((got[0] == 0).all())  # an empty row


@pytest.mark.parametrize("H,cache,q_lora,rank", [(16, None, 0, 640), (12, "fp8_e4m3", 0, 600), (5, None, 160, 1024)])
def test_wide_step_equals_the_general_path(gpu, H, cache, q_lora, rank, monkeypatch):
    """Steps and a short chunk through MLA.forward on the step's own launches
    and on the general path, at tensor and int positions."""
    say(f"wide step H={H} cache={cache} q_lora={q_lora} rank={rank}")
    cfg = MLAConfig(n_embd=512, n_head=H, kv_lora_rank=rank, q_lora_rank=q_lora, max_batch_size=3, max_seq_len=600,
                    bias=H == 12)
    m = MLA(cfg, cache_dtype=cache)
    g = torch.Generator().manual_seed(rank)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if "norm" not in name:
                p.copy_(torch.randn(p.shape, generator=g) * 0.03)
    m.eval().to(BF).to(gpu)
    prompt = torch.randn(3, 500, 512, generator=g).to(BF).to(gpu)
    xs = [torch.randn(3, t, 512, generator=g).to(BF).to(gpu) for t in (1, 1, 9)]
    ragged = torch.tensor([500, 3, 77], dtype=torch.int32, device=gpu)
    outs = {}
    for wide in (True, False):
        calls = []
        real = kernels.merge_project_wide
        monkeypatch.setattr(kernels, "merge_project_wide", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
        if not wide:
            monkeypatch.setattr(MLA, "_wide_step_ok", lambda self, x, n: False)
        m.clear_cache()
        m.set_inference_mode(True)
        with torch.no_grad():
            m.prefill_cache(prompt, 0)
            outs[wide] = [m(xs[0], 500), m(xs[1], ragged), m(xs[2], 501)]
        torch.cuda.synchronize()
        monkeypatch.setattr(kernels, "merge_project_wide", real)
        assert len(calls) == (3 if wide else 0)
    for a, b in zip(outs[True], outs[False]):
        err = (a.double() - b.double()).abs()
        assert not bool((err > 1e-2 + 2e-2 * b.double().abs()).any()), float(err.max())


@pytest.mark.parametrize("rank", [513, 600, 704, 768, 832, 1024])
@pytest.mark.parametrize("fp8", [False, True], ids=["bf16", "e4m3"])
@pytest.mark.parametrize("n_splits,balance", [(1, 0), (5, 0), (40, 256)])
def test_wide_attention_steps(gpu, rank, fp8, n_splits, balance):
    """The channel-split attention against fp64 at the edges of its 32-token
    steps and 16-token tiles, for every spread of channel blocks over the
    waves (NB % 4 = 1, 2, 3, 0), launched three times, to the bounds of
    attn_ref.wide_bars (tests/test_parity_power.py: a lost step breaks them)."""
    say(f"wide attention rank={rank} fp8={fp8} n_splits={n_splits}")
    lens = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 97, 129, 0, 513, 1000, 1999]
    rows, S = len(lens), 2000
    g = torch.Generator(device=gpu).manual_seed(rank + n_splits)
    cache = LatentCache.allocate(rows, S, BF, gpu, fp8=fp8, rank=rank)
    x = torch.randn(rows, S, rank, generator=g, device=gpu)
    if fp8:
        scale = x.abs().amax(-1) / 448
        codes = (x / scale[..., None]).to(torch.float8_e4m3fn)
        cache.ckv[..., :rank] = codes.view(torch.uint8)
        cache.scale.copy_(scale)
        lat = codes.double() * scale.double()[..., None]
    else:
        cache.ckv[..., :rank] = x.to(BF)
        lat = cache.ckv[..., :rank].double()
    cache.kpe.copy_(torch.randn(rows, S, 64, generator=g, device=gpu))
    one, zero = torch.ones(S, 32, dtype=BF, device=gpu), torch.zeros(S, 32, dtype=BF, device=gpu)
    rp = kernels.padded_rank(rank)
    q_abs = (0.5 * torch.randn(rows, 16, rp, generator=g, device=gpu)).to(BF)
    q_pe = torch.randn(rows, 16, 64, generator=g, device=gpu).to(BF)
    sp = torch.tensor(lens, dtype=torch.int32, device=gpu) - 1
    for _ in range(3):
        lse = torch.empty(rows, 16, device=gpu)
        o = kernels.decode_attention(q_abs, q_pe, one, zero, cache, 0.07, start_pos=sp, n_splits=n_splits,
                                     min_chunk=16, lse_out=lse, balance=balance)
        for r, n in enumerate(lens):
            if n == 0:
                assert bool((o[r] == 0).all()) and bool(torch.isneginf(lse[r]).all())
                continue
            s = 0.07 * (q_abs[r, :, :rank].double() @ lat[r, :n].T + q_pe[r].double() @ cache.kpe[r, :n].double().T)
            ref = torch.softmax(s, -1) @ lat[r, :n]
            terms = 0.07 * (q_abs[r, :, :rank].double().abs() @ lat[r, :n].abs().T
                            + q_pe[r].double().abs() @ cache.kpe[r, :n].double().abs().T)
            lim, rms = wide_bars(s, torch.softmax(s, -1), lat[r, :n], ref, terms)
            err = o[r, :, :rank].double() - ref
            assert bool((err.abs() <= lim).all()), (r, n)
            assert bool((err.square().mean(-1, keepdim=True).sqrt() <= rms).all()), (r, n)
            assert float((lse[r].double() - torch.logsumexp(s, -1)).abs().max()) <= 1e-4, (r, n)
            assert bool((o[r, :, rank:] == 0).all())
