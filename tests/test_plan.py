"""Host-side split planning (CPU): how many splits and balanced workgroups a
decode launch asks for, given the workgroups per CU its kernel is built for
(one per CU for the MFMA decode kernel; other counts exercise the formula)."""
from __future__ import annotations

import pytest
import torch

from oracle.mla_ref import MLAConfig
from swamla_amd import kernels
from swamla_amd.mla import MLA


def test_plan_splits_fills_every_slot():
    # config 2: 32 rows over 256 CUs, one workgroup per CU -> 8 splits
    assert kernels.plan_splits(32, 4224, 256) == (8, 256)
    # config 5: 128 rows; three workgroups per CU -> 6 splits, one -> 2
    assert kernels.plan_splits(128, 8256, 256, blocks_per_cu=3) == (6, 256)
    assert kernels.plan_splits(128, 8256, 256, blocks_per_cu=1) == (2, 256)
    # short rows stop at one split per min_chunk tokens
    assert kernels.plan_splits(4, 600, 256, blocks_per_cu=3) == (3, 256)
    assert kernels.plan_splits(0, 100) == (1, 256)


def test_balanced_splits_scale_with_slots():
    assert kernels.balanced_splits(64, 256) == (256, 16)
    assert kernels.balanced_splits(64, 256, blocks_per_cu=3) == (768, 48)
    assert kernels.balanced_splits(200, 256) == (256, 8)
    # more rows than a balanced plan covers, or more rows than slots
    assert kernels.balanced_splits(257, 256, blocks_per_cu=3) == (0, 0)
    assert kernels.balanced_splits(300, 256) == (0, 0)
    assert kernels.balanced_splits(0, 256) == (0, 0)


@pytest.mark.parametrize("cache_dtype,bpc", [(None, 1), ("fp8_e4m3", 3)])
def test_module_plan_uses_workgroups_per_cu(monkeypatch, cache_dtype, bpc):
    """MLA._decode_plan sizes both plans for CUs x the kernel's workgroups per
    CU (the occupancy query needs a GPU, so it is stubbed here with the values
    the GPU tests check)."""
    seen = []

    def fake(dtype, fp8, rank, fused, device):
        seen.append((dtype, fp8, rank, fused))
        return bpc

    monkeypatch.setattr(kernels, "decode_blocks_per_cu", fake)
    m = MLA(MLAConfig(max_batch_size=128, max_seq_len=64), cache_dtype=cache_dtype).to(torch.bfloat16)
    m._num_cus = 256
    ns, mc, bal = m._decode_plan(128, 8256, torch.device("cpu"), False, dtype=torch.bfloat16)
    assert (ns, mc, bal) == (2 * bpc, 256, 0)
    ns, mc, bal = m._decode_plan(64, 8256, torch.device("cpu"), True, dtype=torch.bfloat16)
    assert (ns, bal) == (16 * bpc, 256 * bpc)
    assert seen[0] == (torch.bfloat16, cache_dtype == "fp8_e4m3", 256, True)


def test_packed_blocks_mirrors_the_launcher():
    """kernels.packed_blocks restates launch_linear_packed's grid
    (mla_linear.hip): the decode step's shapes at batch 32 fill the 256 CUs
    once; the stacked input product at 128 rows needs 340 workgroups (two
    slabs of 64 rows x 170 blocks of four octets), wo at 128 rows 256."""
    from swamla_amd import kernels

    assert kernels.packed_blocks(32, 5440, 1024) == 256
    assert kernels.packed_blocks(32, 1024, 2048) == 256
    assert kernels.packed_blocks(64, 5440, 1024) == 256
    assert kernels.packed_blocks(128, 5440, 1024) == 340
    assert kernels.packed_blocks(128, 1024, 2048) == 256
    assert kernels.packed_blocks(1, 8, 512) == 1


def test_committed_traffic_matches_the_current_kernel_source():
    """bench.py copies an HBM traffic figure into its JSON line only from a
    committed profile keyed to the decode kernel's current source; config 2's
    16- and 32-head launches must have one (re-measure after a source change)."""
    import bench

    for heads in (16, 32):
        got = bench.measured_traffic(32, 4224, "bf16", heads=heads)
        assert got is not None and got[0] > 87_000_000, (heads, got)


def test_min_chunk_by_dtype_rank_and_length():
    """The smallest split of a module's decode plan: fixed for bf16 up to rank
    512 and for fp32, growing with sqrt(2 L) above rank 512."""
    f = kernels.min_chunk_for
    assert f(torch.bfloat16, 256, 100) == f(torch.bfloat16, 512, 100000) == 256
    assert f(torch.float32, 256, 1) == f(torch.float32, 1024, 100000) == 16
    wide = [f(torch.bfloat16, 640, n) for n in (0, 1, 576, 2000, 8000, 30000, 1 << 20)]
    assert wide == [32, 32, 32, 64, 128, 240, 256]
    m = MLA(MLAConfig(kv_lora_rank=640, max_batch_size=1, max_seq_len=64)).to(torch.bfloat16)
    m._num_cus = 256
    assert m._split_plan(1, 2000, torch.device("cpu")) == (32, 64)


def test_expansion_groups():
    """Keys and values of a prompt never take more than EXPAND_BYTES: whole
    sequences while they fit, then a sequence's heads in groups (multiples of
    8 where it can be), and none where one head's exceed it."""
    for heads, itemsize in ((16, 2), (32, 2), (12, 4), (5, 2)):
        m = MLA(MLAConfig(n_head=heads, max_batch_size=1, max_seq_len=8))
        for B, L in ((1, 1), (4, 4096), (64, 512), (1, 131072), (3, 200000), (1, 1 << 20), (1, 3 << 20)):
            head = 2 * L * 128 * itemsize
            got = m._expand_groups(B, L, itemsize)
            if head > m.EXPAND_BYTES:
                assert got is None
                continue
            nb, nh = got
            assert nb * nh * head <= m.EXPAND_BYTES and 1 <= nb <= B and 1 <= nh <= heads
            assert nh == heads or (nb == 1 and (nh <= 8 or nh % 8 == 0))
            room = m.EXPAND_BYTES // head
            assert nh > room - 8 if nh < heads else nb == min(B, room // heads)
    m = MLA(MLAConfig(n_head=32, max_batch_size=1, max_seq_len=8))
    assert m._expand_groups(1, 132096, 2) == (1, 7)  # 2.1 GB in one piece


def test_fp32_route_of_prompts():
    """use_expanded_f32 against measured forwards (us expanded / latent): short
    prompts of every head count expand, a few tokens behind a long prefix do
    not, and nothing hangs on one head count or one size."""
    f = kernels.use_expanded_f32
    for heads in (5, 8, 12, 16, 32, 40):
        for rank in (64, 256, 640):
            for B, T in ((1, 2), (1, 64), (2, 160), (1, 320), (1, 321)):
                assert f(B, T, 0, heads, rank), (heads, rank, B, T)
            assert f(1, 64, 2000, heads, rank)  # 176-397 / 168-2834
            assert not f(1, 2, 4000, heads, rank)  # 233-631 / 73-350
    assert f(1, 16, 4000, 12, 256) and not f(1, 8, 4000, 12, 256)  # 275 / 308, 274 / 200


def test_bf16_route_of_prompts():
    """use_expanded on both sides of its crossings, where whole forwards were
    timed on each route (its docstring)."""
    f = kernels.use_expanded
    yes = [(1, 640, 0, 16, 256), (4, 4096, 0, 16, 256), (2, 512, 8192, 16, 256), (8, 1001, 0, 16, 444),
           (4, 2048, 0, 32, 256, True)]
    no = [(1, 256, 0, 16, 256), (1, 512, 0, 16, 256), (32, 64, 1024, 16, 256), (32, 64, 4032, 16, 256), (1, 256, 4096, 16, 256)]
    assert [f(*a) for a in yes] == [True] * len(yes)
    assert [f(*a) for a in no] == [False] * len(no)
