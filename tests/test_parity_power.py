"""The config-scale attention checks can fail: on the CPU, with the fp32
restatement the GPU tests compare against (tests/attn_ref.py), a row of
BASELINE config 4's length that loses or repeats one 64-token tile keeps
o_lat inside the 2e-2 / 1e-2 bar, but moves the log-sum-exp by ~4.9e-4,
beyond the 1e-4 bar tests/test_gpu_configs.py holds the kernels to.  A
zero query's log-sum-exp is log L exactly."""
import math

import pytest
import torch

from attn_ref import LSE_ATOL, H, check, ref_attention_fp32, wide_bars

R, P = 256, 64


def _row(L, seed):
    g = torch.Generator().manual_seed(seed)
    c = torch.randn(L, R, generator=g)
    c[:, 0] = torch.arange(L, dtype=torch.float32) * (8.0 / L) - 4.0  # the GPU tests' position ramp
    c = c.to(torch.bfloat16).float()
    p = torch.randn(L, P, generator=g).to(torch.bfloat16).float()
    q = (0.5 * torch.randn(1, H, R, generator=g)).to(torch.bfloat16)
    qp = (0.5 * torch.randn(1, H, P, generator=g)).to(torch.bfloat16)
    return c, p, q, qp


def _attend(c, p, q, qp):
    L = c.shape[0]
    return ref_attention_fp32(q, qp, lambda r, n: c, lambda r, n: p, [L])


def test_dropped_or_repeated_tile_fails_lse_but_not_o():
    L = 131073
    c, p, q, qp = _row(L, 7)
    o, lse = _attend(c, p, q, qp)
    t0 = 64 * 1000  # one 64-token tile in the middle of the row
    keep = torch.cat([torch.arange(0, t0), torch.arange(t0 + 64, L)])
    rep = torch.cat([torch.arange(0, L), torch.arange(t0, t0 + 64)])
    for name, idx in (("dropped", keep), ("repeated", rep)):
        o2, lse2 = _attend(c[idx], p[idx], q, qp)
        check(o2, o)  # the o_lat bar alone passes ...
        shift = float((lse2 - lse).abs().min())
        assert shift > LSE_ATOL, f"{name} tile: lse moved only {shift:.2e}"  # ... the lse bar does not
        assert abs(shift - 64 / L) < 2e-4, shift


def test_zero_query_lse_is_log_length():
    L = 4097
    c, p, _, _ = _row(L, 8)
    zq, zp = torch.zeros(1, H, R, dtype=torch.bfloat16), torch.zeros(1, H, P, dtype=torch.bfloat16)
    o, lse = _attend(c, p, zq, zp)
    assert float((lse.double() - math.log(L)).abs().max()) < 1e-5
    torch.testing.assert_close(o[0], c.mean(0).expand(H, R), rtol=0, atol=1e-5)


@pytest.mark.parametrize("L", [33, 129, 513, 1000, 1999])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("rank", [513, 1024])
def test_wide_attention_bars_catch_a_lost_step(L, fp8, rank):
    """The bounds test_gpu_wide_step holds the channel-split attention to, on
    its distributions: bf16 weights (rounded twice for e4m3) pass with room,
    and a product that misses the last 32-token step, the last 16-token tile
    or (up to 1,000 tokens) that tile in 64 channels only, fails."""
    g = torch.Generator().manual_seed(L + rank)
    lat, kpe = torch.randn(L, rank, generator=g), torch.randn(L, 64, generator=g)
    q, qp = 0.5 * torch.randn(H, rank, generator=g), torch.randn(H, 64, generator=g)
    bf = lambda t: t.to(torch.bfloat16).double()
    scale = (lat.abs().amax(-1) / 448).double() if fp8 else torch.ones(L, dtype=torch.float64)
    codes = (lat / scale[:, None].float()).to(torch.float8_e4m3fn).double() if fp8 else bf(lat)
    lat, kpe, q, qp = codes * scale[:, None], bf(kpe), bf(q), bf(qp)
    s = 0.07 * (q @ lat.T + qp @ kpe.T)
    p = torch.softmax(s, -1)
    ref = p @ lat
    lim, rms = wide_bars(s, p, lat, ref, 0.07 * (q.abs() @ lat.abs().T + qp.abs() @ kpe.abs().T))

    def within(o):
        err = bf(o) - ref
        return bool((err.abs() <= lim).all()) and bool((err.square().mean(-1, keepdim=True).sqrt() <= rms).all())

    w = bf(torch.exp(s - s.amax(-1, keepdim=True)))  # the weights the product uses
    o = bf(w * scale) @ codes / w.sum(-1, keepdim=True)
    err = (bf(o) - ref).square().mean(-1, keepdim=True).sqrt()
    assert within(o) and bool((2 * err <= rms).all())
    for n in (32, 16):
        lost = w.clone()
        lost[:, L - n:] = 0
        assert not within(bf(lost * scale) @ codes / w.sum(-1, keepdim=True)), n
    part = o.clone()
    part[:, :64] = (bf(lost * scale) @ codes / w.sum(-1, keepdim=True))[:, :64]
    assert not within(part) or L > 1000
