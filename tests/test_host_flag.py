"""The append error flag's memory (CPU: pinned memory and the device wait are
stood in for): a dropped flag's word may still be written by kernels in
flight, so it goes back to the pool only after a wait for its device."""
import copy
import gc
import pickle
import weakref

import pytest
import torch

from swamla_amd import kernels


@pytest.fixture
def flags(monkeypatch):
    """(make a flag, weak references to every word handed out, devices waited for)."""
    words, waits = [], []
    real = torch.zeros

    def zeros(*a, pin_memory=False, **k):
        t = real(*a, **k)
        if pin_memory:
            words.append(weakref.ref(t))
        return t

    def wait(dev):
        assert words[0]() is not None  # still held while the device is waited for
        waits.append(dev)

    monkeypatch.setattr(torch, "zeros", zeros)
    monkeypatch.setattr(torch.cuda, "synchronize", wait)
    monkeypatch.setattr(kernels.HostFlag, "_retired", [])
    return lambda i=0: kernels.HostFlag(torch.device("cuda", i)), words, waits


def test_dropped_flag_is_held_until_its_device_is_waited_for(flags):
    make, words, waits = flags
    a = make(1)
    a._v.value = 1
    assert a.is_set()
    a.clear()
    assert not a.is_set()
    del a
    gc.collect()
    assert words[0]() is not None and waits == []
    b = make(0)
    gc.collect()
    assert words[0]() is None and waits == [torch.device("cuda", 1)]
    assert words[1]() is not None and b.data_ptr() == words[1]().data_ptr()
    make(0)  # nothing of b's was dropped: no wait for it
    assert len(waits) == 1


def test_failed_wait_keeps_the_memory(flags, monkeypatch):
    make, words, _ = flags
    make(0)
    gc.collect()

    def fail(dev):
        raise RuntimeError("busy")

    monkeypatch.setattr(torch.cuda, "synchronize", fail)
    with pytest.raises(RuntimeError):
        make(0)
    gc.collect()
    assert words[0]() is not None


def test_copies_start_without_a_flag(flags):
    make, _, _ = flags
    a = make(0)
    assert copy.deepcopy(a) is None and pickle.loads(pickle.dumps(a)) is None


@pytest.mark.gpu
def test_dropped_flag_is_not_handed_out_again(gpu):
    """In the real pool: no pinned tensor gets a dropped flag's word before
    the next flag is made."""
    flag = kernels.HostFlag(gpu)
    addr = flag.data_ptr()
    del flag
    gc.collect()
    others = [torch.zeros(1, dtype=torch.int32, pin_memory=True) for _ in range(8)]
    assert all(t.data_ptr() != addr for t in others)
    assert any(t.data_ptr() == addr for t, _ in kernels.HostFlag._retired)
    flag = kernels.HostFlag(gpu)
    assert not kernels.HostFlag._retired and not flag.is_set()
