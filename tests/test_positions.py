"""The table an eager step takes its int start_pos from (CPU): made and freed
with the cache, never by a call, and not used for another cache or device."""
import copy

import pytest
import torch

from swamla_amd.kernels import LatentCache
from swamla_amd import MLA, MLAConfig

CPU = torch.device("cpu")


def positions(m, B, start, T=1, cache=None):
    return m._start_positions(B, T, start, cache or m.latent_cache(), CPU)


@pytest.mark.parametrize("cache_dtype", [None, "fp8_e4m3"])
def test_table_lives_with_the_cache(cache_dtype):
    m = MLA(MLAConfig(max_batch_size=3, max_seq_len=11), cache_dtype=cache_dtype)
    assert m._positions is None
    m.set_inference_mode(True)
    tab = m._positions
    assert tab is not None and tuple(tab.shape) == (11, 3)
    for start in (0, 7, 10):
        for B in (1, 3):
            sp = positions(m, B, start)
            assert sp.dtype == torch.int32 and sp.tolist() == [start] * B and sp.is_contiguous()
    assert m._positions is tab  # a call neither makes nor replaces it
    with pytest.raises(ValueError):
        positions(m, 1, 11)
    m.set_inference_mode(False)
    assert m._positions is None
    m.max_batch_size, m.max_seq_len = 5, 20  # a larger cache afterwards
    m.set_inference_mode(True)
    assert positions(m, 5, 19).tolist() == [19] * 5
    m.clear_cache()
    assert m._positions is None


def test_another_cache_takes_a_tensor_of_its_own():
    m = MLA(MLAConfig(max_batch_size=2, max_seq_len=4))
    m.set_inference_mode(True)
    big = LatentCache.allocate(3, 9, torch.float32, CPU)
    assert positions(m, 3, 8, cache=big).tolist() == [8] * 3
    tab = m._positions
    sp = positions(m, 2, 1, T=3)  # prompts and chunks: a tensor of their own
    assert sp.tolist() == [1, 1] and sp.untyped_storage().data_ptr() != tab.untyped_storage().data_ptr()
    m._positions = torch.zeros(9, 2, dtype=torch.int32, device="meta")  # the table of a module since moved
    assert positions(m, 2, 3).tolist() == [3, 3]


def test_copies_have_tables_of_their_own():
    m = MLA(MLAConfig(max_batch_size=2, max_seq_len=4))
    m.set_inference_mode(True)
    c = copy.deepcopy(m)
    m.set_inference_mode(False)
    assert positions(c, 2, 3).tolist() == [3, 3]
